// k_gemv_f.hip -- float-dot GEMV for the weight types without a vec_dot kernel: F32, F16,
// Q4_1, Q5_1, Q8_1, Q2_K and Q3_K (larger batches take k_gemm_f.hip, with the same decoders).
//
// The reference routes these through the fallback of matmul_quant (src/core/quant.cpp:
// 1404-1430; matmul_quant_batch runs it row by row, 1471-1474): each weight row is
// dequantized to fp32 and dotted with the fp32 activation row, which is NOT quantized to
// Q8_0. So here
//     y[t, j] = bias[j] + sum_i x[t, i] * deq(W[j, i])
// in fp32. F32 and F16 take one fma per element and activation row. The quantized types
// dequantize as w = A q + B over groups of 16 or 32 elements (q the element's small
// non-negative or int8 code, A and B the group's scale and offset as the reference's deq_*
// functions form them, quant.cpp:28-298), so the dot is regrouped per group:
//     sum_i x_i w_i = A * sum_i x_i q_i + B * sum_i x_i,
// one fma per element on the exact code, then two per group; the group sums of x are formed
// once, with the activation rows' staging. Only the rounding order differs from the
// reference (an exact product per element, a few roundings per group of 16 or 32): lanes own
// 32-element units of a row and the partial sums are added across lanes.
//
// Work split. A unit is 32 consecutive elements of a row: 32 fp32 or fp16 values, one
// Q4_1 / Q5_1 / Q8_1 block, or one eighth of a Q2_K / Q3_K super-block. A row's units are
// spread over L lanes (L = 64, or the power of two covering the units of a short row, so a
// wave then works on 64 / L rows at once); each lane loads the raw bytes of two units before
// decoding the first, and many waves per CU keep the HBM stream busy.
//
// Activations. The MR activation rows of a workgroup's token group are staged in LDS as fp32
// with 16 bytes of padding after every 32 values, so the 16-byte reads of the lanes (units at
// a stride of 144 bytes) spread over all 64 banks, followed by the rows' sums of every 16
// values (for the grouped types). Rows too long for the LDS budget (80 KB, two workgroups per
// CU) are read from global memory instead (they stay in L2), and the quantized types then
// take the per-element form: decode w, one fma per element.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device_utils.h"
#include "float_units.h"
#include "ggml_blocks.h"
#include "launch.h"

namespace cllm_hip {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr size_t kLdsBudget = 80 * 1024;  // two workgroups per CU

// ------------------------------------------------------------------------------ kernel


__host__ __device__ constexpr int xpad_row(int k) { return k + k / 8; }  // floats per LDS row

// Types whose dot is regrouped per 32 elements (gdot), from the LDS-staged activations.
// Q2_K and Q3_K keep the per-element form: regrouped per 16 elements they measured no faster
// on one activation row at 14336 x 4096 (Q2_K 12.6 us either way; Q3_K 15.8, with whole
// half-super-block items per lane 14.1) and, as half-super-block items, slower on four
// (63 / 65 us against 52 / 56). A batch row and the same row alone must take one path.
__host__ __device__ constexpr bool grouped(uint32_t T) {
    return T == T_Q4_1 || T == T_Q5_1 || T == T_Q8_1;
}
// LDS floats per staged activation row: the padded row, and the sums of its 16-value groups
__host__ __device__ constexpr int xlds_row(uint32_t T, int k) { return xpad_row(k) + (grouped(T) ? k / 16 : 0); }

// Workgroups per CU of the pipelined kernel for one activation row, 0 where the per-row
// kernel is faster (MI355X, 14336 x 4096, cold weights, us, per-row kernel against the
// pipelined one at 3 / 4 / 8 workgroups per CU: Q4_1 12.9 against 12.4 / 11.7 / 12.3, Q5_1
// 14.2 against 13.8 / 13.5 / 14.1; Q8_1 15.3 against 15.5 / 15.9 / 16.2)
template <uint32_t T>
constexpr int fp_wgs_per_cu() {
    return T == T_Q4_1 || T == T_Q5_1 ? 4 : 0;
}

template <int MR>
__device__ __forceinline__ void fma_unit(const float (&w)[32], const float* xp, int xstride,
                                         float (&acc)[MR]) {
#pragma unroll
    for (int t = 0; t < MR; ++t) {
        const float4* p = (const float4*)(xp + (size_t)t * xstride);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const float4 xv = p[q];
            acc[t] = __builtin_fmaf(xv.x, w[4 * q], acc[t]);
            acc[t] = __builtin_fmaf(xv.y, w[4 * q + 1], acc[t]);
            acc[t] = __builtin_fmaf(xv.z, w[4 * q + 2], acc[t]);
            acc[t] = __builtin_fmaf(xv.w, w[4 * q + 3], acc[t]);
        }
    }
}

// Stages the MR activation rows from t0 (zeros past m) in LDS with the 16-byte pad per 32
// values; with GS a quad of lanes (16 consecutive values, never across rows: k / 4 is a
// multiple of 4) also forms the group's sum, in a fixed order, into xg[t][k / 16]. Ends with
// a workgroup barrier.
template <int MR, bool GS, int NT = kThreads>
__device__ __forceinline__ void stage_rows(const float* __restrict__ x, int k, int m, int t0, float* xs,
                                           float* xg) {
    const int q4 = k / 4;
    const int srow = xpad_row(k), gstride = k / 16;
    for (int i = threadIdx.x; i < MR * q4; i += NT) {
        const int t = i / q4, e = 4 * (i - t * q4);
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (t0 + t < m) v = *(const float4*)(x + (size_t)(t0 + t) * k + e);
        *(float4*)(xs + t * srow + e + (e >> 5) * 4) = v;
        if constexpr (GS) {
            float p = (v.x + v.y) + (v.z + v.w);
            p += dpp_f32<DPP_QUAD_SWAP1>(p);
            p += dpp_f32<DPP_QUAD_SWAP2>(p);
            if ((i & 3) == 0) xg[t * gstride + (e >> 4)] = p;
        }
    }
    __syncthreads();
}

// grid (row workgroups, token groups of MR), NT threads. lpr_log2 = log2(lanes per row).
template <uint32_t T, int MR, bool XG, int NT = kThreads>
__global__ __launch_bounds__(NT) void k_gemv_f(const uint8_t* __restrict__ w,
                                                     size_t row_bytes, int k, int n, int m,
                                                     const float* __restrict__ x,
                                                     const float* __restrict__ bias,
                                                     float* __restrict__ y, int lpr_log2) {
    using U = FUnit<T>;
    constexpr bool GDOT = grouped(T) && !XG;
    extern __shared__ __align__(16) float xs[];
    const int t0 = blockIdx.y * MR;
    const int units = k / 32;
    const int srow = xpad_row(k);
    const int gstride = k / 16;
    float* xg = xs + MR * srow;  // GDOT: [t][k / 16] sums of 16 activations
    if constexpr (!XG) stage_rows<MR, GDOT, NT>(x, k, m, t0, xs, xg);
    const int lane = threadIdx.x & 63;
    const int lpr = 1 << lpr_log2;
    const int sub = lane & (lpr - 1);
    const int rpw = 64 >> lpr_log2;  // rows per wave
    const int gw = blockIdx.x * (NT / 64) + (threadIdx.x >> 6);
    const int nw = gridDim.x * (NT / 64);
    // activation source: LDS rows, or global rows clamped to the last valid one
    const float* xbase = XG ? x + (size_t)min(t0, m - 1) * k : xs;
    const int xstride = XG ? k : srow;
    auto xptr = [&](int u) { return XG ? xbase + 32 * u : xbase + 36 * u; };

    for (int rb = gw * rpw; rb < n; rb += nw * rpw) {
        const int j = rb + (lane >> lpr_log2);
        const uint8_t* row = w + (size_t)min(j, n - 1) * row_bytes;
        float acc[MR];
#pragma unroll
        for (int t = 0; t < MR; ++t) acc[t] = 0.0f;
        if constexpr (GDOT) {
            // each lane two units at a time. Both units' loads go out before either is used:
            // when some lane of the wave has a second unit (u - sub is wave-uniform), every
            // lane computes one (a lane without one takes unit u again and keeps its sums).
            // Under a per-lane branch the second unit's loads would be issued after the first
            // one's arithmetic, and each row would take two round trips.
            for (int u = sub; u < units; u += 2 * lpr) {
                const bool two = u + lpr < units;
                if (u - sub + lpr < units) {
                    const int u1 = two ? u + lpr : u;
                    const typename U::Raw r0 = U::load(row, u);
                    const typename U::Raw r1 = U::load(row, u1);
                    U::template gdot<MR>(r0, u, xptr(u), xstride, xg + 2 * u, gstride, acc);
                    float acc1[MR];
#pragma unroll
                    for (int t = 0; t < MR; ++t) acc1[t] = acc[t];
                    U::template gdot<MR>(r1, u1, xptr(u1), xstride, xg + 2 * u1, gstride, acc1);
#pragma unroll
                    for (int t = 0; t < MR; ++t) acc[t] = two ? acc1[t] : acc[t];
                } else {
                    U::template gdot<MR>(U::load(row, u), u, xptr(u), xstride, xg + 2 * u, gstride, acc);
                }
            }
        } else {
            for (int u = sub; u < units; u += 2 * lpr) {
                const bool two = u + lpr < units;
                const typename U::Raw r0 = U::load(row, u);
                const typename U::Raw r1 = U::load(row, two ? u + lpr : u);
                float wv[32];
                U::decode(r0, u, wv);
                fma_unit<MR>(wv, xptr(u), xstride, acc);
                if (two) {
                    U::decode(r1, u + lpr, wv);
                    fma_unit<MR>(wv, xptr(u + lpr), xstride, acc);
                }
            }
        }
#pragma unroll
        for (int t = 0; t < MR; ++t)
            for (int off = lpr >> 1; off > 0; off >>= 1) acc[t] += __shfl_xor(acc[t], off, 64);
        if (sub == 0 && j < n) {
            const float b = bias ? bias[j] : 0.0f;
#pragma unroll
            for (int t = 0; t < MR; ++t)
                if (t0 + t < m) y[(size_t)(t0 + t) * n + j] = acc[t] + b;
        }
    }
}

// The grouped types on rows of at most two units per lane, activations in LDS (staged as for
// k_gemv_f). Each wave walks rows rb, rb + step, .. and issues the next row's loads before
// the current row's arithmetic, unconditionally (rows past the matrix read the last row
// again, units past a short row the last unit), so that a wave keeps a row of loads in
// flight while it computes. (k_gemv_f gives every wave about one row at these sizes: the
// whole matrix is requested at once and no arithmetic overlaps the transfer.) The per-row
// arithmetic is k_gemv_f's, in the same order, so the two kernels agree bit for bit.
// grid (row workgroups, token groups of MR), 256 threads.
template <uint32_t T, int MR>
__global__ __launch_bounds__(kThreads) void k_gemv_fp(const uint8_t* __restrict__ w,
                                                      size_t row_bytes, int k, int n, int m,
                                                      const float* __restrict__ x,
                                                      const float* __restrict__ bias,
                                                      float* __restrict__ y, int lpr_log2) {
    using U = FUnit<T>;
    static_assert(grouped(T), "the grouped types only");
    extern __shared__ __align__(16) float xs[];
    const int t0 = blockIdx.y * MR;
    const int srow = xpad_row(k);
    const int gstride = k / 16;
    float* xg = xs + MR * srow;
    stage_rows<MR, true>(x, k, m, t0, xs, xg);

    const int lane = threadIdx.x & 63;
    const int lpr = 1 << lpr_log2;
    const int sub = lane & (lpr - 1);
    const int rpw = 64 >> lpr_log2;
    const int step = (int)gridDim.x * kWaves * rpw;
    const int units = k / 32;
    const bool has0 = sub < units, has1 = sub + lpr < units;
    const int u0 = min(sub, units - 1), u1 = min(sub + lpr, units - 1);
    auto row_at = [&](int rb) {
        return w + (size_t)min(rb + (lane >> lpr_log2), n - 1) * row_bytes;
    };
    const int rb0 = (blockIdx.x * kWaves + (threadIdx.x >> 6)) * rpw;
    if (rb0 >= n) return;  // wave-uniform, after the last barrier
    // NI units per lane (2 when some lane's row has a second one, else 1: uniform)
    auto walk = [&]<int NI>() {
        typename U::Raw a0 = U::load(row_at(rb0), u0);
        typename U::Raw a1 = U::load(row_at(rb0), NI == 2 ? u1 : u0);
        for (int rb = rb0; rb < n; rb += step) {
            const typename U::Raw c0 = a0;
            const typename U::Raw c1 = a1;
            a0 = U::load(row_at(rb + step), u0);
            if constexpr (NI == 2) a1 = U::load(row_at(rb + step), u1);
            float acc[MR], acc1[MR];
#pragma unroll
            for (int t = 0; t < MR; ++t) acc[t] = 0.0f;
            U::template gdot<MR>(c0, u0, xs + 36 * u0, srow, xg + 2 * u0, gstride, acc);
            if constexpr (NI == 2) {
#pragma unroll
                for (int t = 0; t < MR; ++t) acc1[t] = acc[t];
                U::template gdot<MR>(c1, u1, xs + 36 * u1, srow, xg + 2 * u1, gstride, acc1);
            }
#pragma unroll
            for (int t = 0; t < MR; ++t) acc[t] = (NI == 2 && has1) ? acc1[t] : (has0 ? acc[t] : 0.0f);
#pragma unroll
            for (int t = 0; t < MR; ++t)
                for (int off = lpr >> 1; off > 0; off >>= 1) acc[t] += __shfl_xor(acc[t], off, 64);
            const int j = rb + (lane >> lpr_log2);
            if (sub == 0 && j < n) {
                const float b = bias ? bias[j] : 0.0f;
#pragma unroll
                for (int t = 0; t < MR; ++t)
                    if (t0 + t < m) y[(size_t)(t0 + t) * n + j] = acc[t] + b;
            }
        }
    };
    if (lpr < units)
        walk.template operator()<2>();
    else
        walk.template operator()<1>();
}

// F32 / F16 rows whose length is not a multiple of 32: one wave per row, lanes stride over
// the elements, activations from global memory, every token of the batch in turn.
template <uint32_t T>
__global__ __launch_bounds__(kThreads) void k_gemv_f_any(const uint8_t* __restrict__ w,
                                                         size_t row_bytes, int k, int n, int m,
                                                         const float* __restrict__ x,
                                                         const float* __restrict__ bias,
                                                         float* __restrict__ y) {
    const int lane = threadIdx.x & 63;
    const int gw = blockIdx.x * kWaves + (threadIdx.x >> 6);
    const int nw = gridDim.x * kWaves;
    for (int j = gw; j < n; j += nw) {
        const uint8_t* row = w + (size_t)j * row_bytes;
        for (int t = 0; t < m; ++t) {
            const float* xt = x + (size_t)t * k;
            float acc = 0.0f;
            for (int e = lane; e < k; e += 64) {
                const float wv = T == T_F32 ? ((const float*)row)[e]
                                            : f16_to_f32(((const uint16_t*)row)[e]);
                acc = __builtin_fmaf(xt[e], wv, acc);
            }
            acc = wave_sum(acc);
            if (lane == 0) y[(size_t)t * n + j] = acc + (bias ? bias[j] : 0.0f);
        }
    }
}

int device_cus_f() {
    static int cus = 0;
    if (cus == 0) {
        int dev = 0, v = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0)
            cus = v;
        else
            cus = 256;
    }
    return cus;
}

template <uint32_t T, int MR, bool XG>
hipError_t launch_mr(const uint8_t* w, size_t row_bytes, int k, int n, int m, const float* x,
                     const float* bias, float* y, hipStream_t stream) {
    const int units = k / 32;
    int lpr_log2 = 6;
    while (lpr_log2 > 0 && (1 << (lpr_log2 - 1)) >= units) --lpr_log2;
    const int rpw = 64 >> lpr_log2;
    const int64_t row_groups = ((int64_t)n + rpw - 1) / rpw;
    const int64_t wgs = std::min<int64_t>((row_groups + kWaves - 1) / kWaves,
                                          (int64_t)device_cus_f() * 8);
    const int groups = (m + MR - 1) / MR;
    if (groups > 65535) return hipErrorInvalidConfiguration;
    const size_t lds = XG ? 0 : (size_t)MR * xlds_row(T, k) * sizeof(float);
    if constexpr (grouped(T) && !XG && MR == 1) {
        // rows of at most two units per lane take the pipelined kernel where it is the
        // faster one, on fp_wgs_per_cu workgroups per CU (fewer if the rows run out). The
        // tuning knob "gemv_fp_wgs" forces it at 1 to 8 workgroups per CU, or (9) the per-row
        // kernel.
        const int knob = tuning().gemv_fp_wgs.load(std::memory_order_relaxed);
        const int per_cu = knob == 0 ? fp_wgs_per_cu<T>() : knob == 9 ? 0 : knob;
        if (units <= 2 * (1 << lpr_log2) && per_cu > 0) {
            const int64_t fwgs = std::min<int64_t>((row_groups + kWaves - 1) / kWaves,
                                                   (int64_t)device_cus_f() * per_cu);
            hipLaunchKernelGGL((k_gemv_fp<T, MR>), dim3((unsigned)fwgs, (unsigned)groups),
                               dim3(kThreads), lds, stream, w, row_bytes, k, n, m, x, bias, y, lpr_log2);
            return hipGetLastError();
        }
    }
    if constexpr (MR >= 2 && !XG) {
        // Several activation rows whose staging takes more than 20 KB of LDS run on 1024-thread
        // workgroups. LDS then holds fewer than eight 256-thread workgroups per CU (four rows
        // of 4096, ~78 KB: two), which left each wave's row loads exposed (MI355X, 14336 x
        // 4096 at 4 rows, cold weights, us, 256 / 1024 threads: Q2_K 51.3 / 21.8, Q4_1 50.5 /
        // 25.8, Q8_1 54.6 / 28.3, F16 56.4 / 32.9, F32 78.2 / 57.7). Shorter rows keep 256
        // threads (the F16 151936 x 896 head at 4 rows, 16 KB: 61.9 against 78.4 us). The
        // grid is the workgroups resident at once (two per CU; waves walk further rows): more
        // would restage the rows in every later workgroup. Same bits either way: a row's
        // additions do not depend on the workgroup size.
        if (lds > 20 * 1024) {
            constexpr int NT = 1024;
            const int64_t wgs_nt = std::min<int64_t>((row_groups + NT / 64 - 1) / (NT / 64),
                                                     (int64_t)device_cus_f() * 2);
            hipLaunchKernelGGL((k_gemv_f<T, MR, XG, NT>), dim3((unsigned)wgs_nt, (unsigned)groups),
                               dim3(NT), lds, stream, w, row_bytes, k, n, m, x, bias, y, lpr_log2);
            return hipGetLastError();
        }
    }
    hipLaunchKernelGGL((k_gemv_f<T, MR, XG>), dim3((unsigned)wgs, (unsigned)groups),
                       dim3(kThreads), lds, stream, w, row_bytes, k, n, m, x, bias, y, lpr_log2);
    return hipGetLastError();
}

template <uint32_t T>
hipError_t launch_type(const uint8_t* w, int k, int n, int m, const float* x, const float* bias,
                       float* y, hipStream_t stream) {
    const size_t row_bytes = (size_t)(k / block_elems(T)) * block_bytes(T);
    if constexpr (T == T_F32 || T == T_F16) {
        if (k % 32 != 0) {
            const int64_t wgs = std::min<int64_t>(((int64_t)n + kWaves - 1) / kWaves,
                                                  (int64_t)device_cus_f() * 8);
            hipLaunchKernelGGL((k_gemv_f_any<T>), dim3((unsigned)wgs), dim3(kThreads), 0, stream,
                               w, row_bytes, k, n, m, x, bias, y);
            return hipGetLastError();
        }
    }
    const size_t row_lds = (size_t)xlds_row(T, k) * sizeof(float);
    if (m >= 3 && 4 * row_lds <= kLdsBudget)
        return launch_mr<T, 4, false>(w, row_bytes, k, n, m, x, bias, y, stream);
    if (m >= 2 && 2 * row_lds <= kLdsBudget)
        return launch_mr<T, 2, false>(w, row_bytes, k, n, m, x, bias, y, stream);
    if (row_lds <= kLdsBudget)
        return launch_mr<T, 1, false>(w, row_bytes, k, n, m, x, bias, y, stream);
    if (m >= 3) return launch_mr<T, 4, true>(w, row_bytes, k, n, m, x, bias, y, stream);
    return launch_mr<T, 1, true>(w, row_bytes, k, n, m, x, bias, y, stream);
}

// Rows ids[i] of a weight matrix dequantized to fp32 (get_embedding's dequantize_block,
// engine.cpp:310-317, quant.cpp:371-389): one thread per 32-element unit.
template <uint32_t T>
__global__ __launch_bounds__(kThreads) void k_dequant_rows(const uint8_t* __restrict__ w,
                                                           size_t row_bytes, int k,
                                                           const int32_t* __restrict__ ids,
                                                           int n_ids, float* __restrict__ out) {
    const int units = k / 32;
    const int64_t g = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (g >= (int64_t)n_ids * units) return;
    const int r = (int)(g / units), u = (int)(g - (int64_t)r * units);
    float v[32];
    FUnit<T>::decode(FUnit<T>::load(w + (size_t)ids[r] * row_bytes, u), u, v);
    f32x4* o = (f32x4*)(out + (size_t)r * k + 32 * u);
#pragma unroll
    for (int q = 0; q < 8; ++q) o[q] = f32x4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
}

// F32 / F16 rows of any length, one element per thread.
template <uint32_t T>
__global__ __launch_bounds__(kThreads) void k_dequant_rows_any(const uint8_t* __restrict__ w,
                                                               size_t row_bytes, int k,
                                                               const int32_t* __restrict__ ids,
                                                               int n_ids, float* __restrict__ out) {
    const int64_t g = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (g >= (int64_t)n_ids * k) return;
    const int r = (int)(g / k), e = (int)(g - (int64_t)r * k);
    const uint8_t* row = w + (size_t)ids[r] * row_bytes;
    out[(size_t)r * k + e] = T == T_F32 ? ((const float*)row)[e] : f16_to_f32(((const uint16_t*)row)[e]);
}

// binary16 bits -> float by integer operations only: exact for every encoding, and a NaN keeps
// its payload and signalling bit (half_to_float, include/cllm/core/quant.hpp:31-56), which the
// hardware conversion would quiet.
__device__ __forceinline__ float f16_to_f32_exact(uint32_t h) {
    const uint32_t sign = (h & 0x8000u) << 16, e = (h >> 10) & 0x1Fu, man = h & 0x3FFu;
    if (e == 0x1Fu) return __builtin_bit_cast(float, sign | 0x7F800000u | (man << 13));
    if (e != 0) return __builtin_bit_cast(float, sign | ((e + 112u) << 23) | (man << 13));
    // zero or subnormal: man * 2^-24, exact in fp32
    return __builtin_bit_cast(float, sign | __builtin_bit_cast(uint32_t, (float)man * 0x1p-24f));
}

// float -> binary16 bits by the rule of the reference header's float_to_half (its
// include/cllm/core/quant.hpp:58-87): results in the normal range keep the top 10 mantissa
// bits (truncation), results below it are rounded to nearest with ties to even, results
// below 2^-25 or so become signed zero, overflow becomes infinity and NaN a quiet NaN.
__device__ __forceinline__ uint32_t f32_to_f16_trunc(float f) {
    const uint32_t x = __builtin_bit_cast(uint32_t, f);
    const uint32_t sign = (x >> 16) & 0x8000u;
    const uint32_t biased = (x >> 23) & 0xFFu;
    uint32_t man = x & 0x7FFFFFu;
    if (biased == 0xFFu) return sign | (man ? 0x7E00u : 0x7C00u);
    const int e = (int)biased - 112;  // rebias 127 -> 15
    if (e >= 31) return sign | 0x7C00u;
    if (e > 0) return sign | ((uint32_t)e << 10) | (man >> 13);
    if (e < -10) return sign;
    man |= 0x800000u;
    const uint32_t shift = (uint32_t)(14 - e);
    return sign | ((man + ((1u << (shift - 1)) - 1u) + ((man >> shift) & 1u)) >> shift);
}

// Elements [0, n) of a run of blocks (dequantize_block, quant.cpp:371-389, and
// dequantize_block_f16, 398-407): thread u decodes the 32-element unit u; the elements at and
// past n of a partial last block are not written, as the reference's loops guard them. H: the
// values go out as binary16 bits (f32_to_f16_trunc) instead of fp32.
template <uint32_t T, bool H>
__global__ __launch_bounds__(kThreads) void k_dequant_span(const uint8_t* __restrict__ src,
                                                           int64_t n, float* __restrict__ out,
                                                           uint16_t* __restrict__ out16) {
    const int64_t u = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (u >= (n + 31) / 32) return;
    float v[32];
    if constexpr (T == T_F16) {
        // integer conversion, so NaN payloads pass unchanged as in half_to_float
        const u32x4* p = (const u32x4*)(src + 64 * u);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const u32x4 r = p[q];
            const uint32_t d[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                v[8 * q + 2 * i] = f16_to_f32_exact(d[i] & 0xFFFFu);
                v[8 * q + 2 * i + 1] = f16_to_f32_exact(d[i] >> 16);
            }
        }
    } else {
        FUnit<T>::decode(FUnit<T>::load(src, (int)u), (int)u, v);
    }
    const int64_t e0 = 32 * u;
    if (e0 + 32 <= n) {
        if constexpr (H) {
            u32x4* o = (u32x4*)(out16 + e0);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                uint32_t p[4];
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    p[i] = f32_to_f16_trunc(v[8 * q + 2 * i]) | (f32_to_f16_trunc(v[8 * q + 2 * i + 1]) << 16);
                o[q] = u32x4{p[0], p[1], p[2], p[3]};
            }
        } else {
            f32x4* o = (f32x4*)(out + e0);
#pragma unroll
            for (int q = 0; q < 8; ++q) o[q] = f32x4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
        }
    } else {
#pragma unroll
        for (int i = 0; i < 32; ++i) {
            if (e0 + i < n) {
                if constexpr (H)
                    out16[e0 + i] = (uint16_t)f32_to_f16_trunc(v[i]);
                else
                    out[e0 + i] = v[i];
            }
        }
    }
}

// F32 / F16 runs of any length, one element per thread.
template <uint32_t T, bool H>
__global__ __launch_bounds__(kThreads) void k_dequant_span_any(const uint8_t* __restrict__ src,
                                                               int64_t n, float* __restrict__ out,
                                                               uint16_t* __restrict__ out16) {
    const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (i >= n) return;
    const float v = T == T_F32 ? ((const float*)src)[i] : f16_to_f32_exact(((const uint16_t*)src)[i]);
    if constexpr (H)
        out16[i] = (uint16_t)f32_to_f16_trunc(v);
    else
        out[i] = v;
}

template <uint32_t T>
hipError_t launch_span_t(const uint8_t* src, int64_t n, float* out, uint16_t* out16,
                         hipStream_t stream) {
    if ((T == T_F32 || T == T_F16) && n % 32 != 0) {
        const unsigned grid = (unsigned)((n + kThreads - 1) / kThreads);
        if (out16)
            hipLaunchKernelGGL((k_dequant_span_any<T, true>), dim3(grid), dim3(kThreads), 0, stream, src, n, out, out16);
        else
            hipLaunchKernelGGL((k_dequant_span_any<T, false>), dim3(grid), dim3(kThreads), 0, stream, src, n, out, out16);
    } else {
        const unsigned grid = (unsigned)(((n + 31) / 32 + kThreads - 1) / kThreads);
        if (out16)
            hipLaunchKernelGGL((k_dequant_span<T, true>), dim3(grid), dim3(kThreads), 0, stream, src, n, out, out16);
        else
            hipLaunchKernelGGL((k_dequant_span<T, false>), dim3(grid), dim3(kThreads), 0, stream, src, n, out, out16);
    }
    return hipGetLastError();
}

template <uint32_t T>
hipError_t launch_dequant_t(const uint8_t* w, int k, const int32_t* ids, int n, float* out,
                            hipStream_t stream) {
    const size_t row_bytes = (size_t)(k / block_elems(T)) * block_bytes(T);
    if ((T == T_F32 || T == T_F16) && k % 32 != 0) {
        const int64_t threads = (int64_t)n * k;
        hipLaunchKernelGGL((k_dequant_rows_any<T>), dim3((unsigned)((threads + kThreads - 1) / kThreads)),
                           dim3(kThreads), 0, stream, w, row_bytes, k, ids, n, out);
    } else {
        const int64_t threads = (int64_t)n * (k / 32);
        hipLaunchKernelGGL((k_dequant_rows<T>), dim3((unsigned)((threads + kThreads - 1) / kThreads)),
                           dim3(kThreads), 0, stream, w, row_bytes, k, ids, n, out);
    }
    return hipGetLastError();
}

}  // namespace

hipError_t launch_dequantize_rows(uint32_t type, const uint8_t* w, int k, const int32_t* ids,
                                  int n, float* out, hipStream_t stream) {
    if (n <= 0) return hipSuccess;
    if (k <= 0 || k % block_elems(type) != 0) return hipErrorInvalidValue;
    switch (type) {
        case T_F32: return launch_dequant_t<T_F32>(w, k, ids, n, out, stream);
        case T_F16: return launch_dequant_t<T_F16>(w, k, ids, n, out, stream);
        case T_Q4_0: return launch_dequant_t<T_Q4_0>(w, k, ids, n, out, stream);
        case T_Q4_1: return launch_dequant_t<T_Q4_1>(w, k, ids, n, out, stream);
        case T_Q5_0: return launch_dequant_t<T_Q5_0>(w, k, ids, n, out, stream);
        case T_Q5_1: return launch_dequant_t<T_Q5_1>(w, k, ids, n, out, stream);
        case T_Q8_0: return launch_dequant_t<T_Q8_0>(w, k, ids, n, out, stream);
        case T_Q8_1: return launch_dequant_t<T_Q8_1>(w, k, ids, n, out, stream);
        case T_Q2_K: return launch_dequant_t<T_Q2_K>(w, k, ids, n, out, stream);
        case T_Q3_K: return launch_dequant_t<T_Q3_K>(w, k, ids, n, out, stream);
        case T_Q4_K: return launch_dequant_t<T_Q4_K>(w, k, ids, n, out, stream);
        case T_Q5_K: return launch_dequant_t<T_Q5_K>(w, k, ids, n, out, stream);
        case T_Q6_K: return launch_dequant_t<T_Q6_K>(w, k, ids, n, out, stream);
        default: return hipErrorNotSupported;
    }
}

hipError_t launch_dequantize_span(uint32_t type, const uint8_t* src, int64_t n, float* out,
                                  uint16_t* out16, hipStream_t stream) {
    if (n <= 0) return hipSuccess;
    if ((out == nullptr) == (out16 == nullptr) || n > ((int64_t)1 << 36)) return hipErrorInvalidValue;
    switch (type) {
        case T_F32: return launch_span_t<T_F32>(src, n, out, out16, stream);
        case T_F16: return launch_span_t<T_F16>(src, n, out, out16, stream);
        case T_Q4_0: return launch_span_t<T_Q4_0>(src, n, out, out16, stream);
        case T_Q4_1: return launch_span_t<T_Q4_1>(src, n, out, out16, stream);
        case T_Q5_0: return launch_span_t<T_Q5_0>(src, n, out, out16, stream);
        case T_Q5_1: return launch_span_t<T_Q5_1>(src, n, out, out16, stream);
        case T_Q8_0: return launch_span_t<T_Q8_0>(src, n, out, out16, stream);
        case T_Q8_1: return launch_span_t<T_Q8_1>(src, n, out, out16, stream);
        case T_Q2_K: return launch_span_t<T_Q2_K>(src, n, out, out16, stream);
        case T_Q3_K: return launch_span_t<T_Q3_K>(src, n, out, out16, stream);
        case T_Q4_K: return launch_span_t<T_Q4_K>(src, n, out, out16, stream);
        case T_Q5_K: return launch_span_t<T_Q5_K>(src, n, out, out16, stream);
        case T_Q6_K: return launch_span_t<T_Q6_K>(src, n, out, out16, stream);
        default: return hipErrorNotSupported;
    }
}

bool gemv_f_supported(uint32_t type) {
    return type == T_F32 || type == T_F16 || type == T_Q4_1 || type == T_Q5_1 ||
           type == T_Q8_1 || type == T_Q2_K || type == T_Q3_K;
}

hipError_t launch_gemv_f(uint32_t type, const uint8_t* w, int k, int n, int m, const float* x,
                         const float* bias, float* y, hipStream_t stream) {
    if (n <= 0 || m <= 0) return hipSuccess;
    if (k <= 0 || k % block_elems(type) != 0) return hipErrorInvalidValue;
    if (gemm_f_takes(type, k, n, m)) return launch_gemm_f(type, w, k, n, m, x, bias, y, stream);
    switch (type) {
        case T_F32: return launch_type<T_F32>(w, k, n, m, x, bias, y, stream);
        case T_F16: return launch_type<T_F16>(w, k, n, m, x, bias, y, stream);
        case T_Q4_1: return launch_type<T_Q4_1>(w, k, n, m, x, bias, y, stream);
        case T_Q5_1: return launch_type<T_Q5_1>(w, k, n, m, x, bias, y, stream);
        case T_Q8_1: return launch_type<T_Q8_1>(w, k, n, m, x, bias, y, stream);
        case T_Q2_K: return launch_type<T_Q2_K>(w, k, n, m, x, bias, y, stream);
        case T_Q3_K: return launch_type<T_Q3_K>(w, k, n, m, x, bias, y, stream);
        default: return hipErrorNotSupported;
    }
}

}  // namespace cllm_hip
