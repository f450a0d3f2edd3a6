// k_gemm_f.hip -- float-dot GEMM for batches of the weight types without a vec_dot kernel
// (F32, F16, Q4_1, Q5_1, Q8_1, Q2_K, Q3_K), on bf16 MFMA with fp32's precision.
//
// The reference dequantizes a weight row to fp32 and dots it with the fp32 activation rows
// (src/core/quant.cpp:1404-1430, matmul_quant_batch 1471-1474). The GEMV kernels
// (k_gemv_f.hip) do that with one FMA per weight and row and read the matrix once per 4 rows,
// which 301 rows of a 4096 x 4096 Q3_K matrix turned into 437 us of VALU work at 23 TFLOP/s;
// here they take 67 us (150 TFLOP/s), bound by the decoding and splitting VALU work beside the
// MFMAs and by each wave's serial path through a stage, two waves to a SIMD.
//
// Split operands. An fp32 value is the sum of three bf16 values of 8 significant bits
// (rounded to nearest, so the three cover 26 bits), and a bf16 product is exact in the MFMA's
// fp32 accumulator. With w = w0 + w1 + w2 and x = x0 + x1 + x2, the six products w0 x0, w0 x1,
// w0 x2, w1 x0, w1 x1, w2 x0 leave out w1 x2 and w2 x1, up to 2^-25 of the product each: at most
// what rounding an fp32 product takes off (2^-24), and far less on average. At 16 times the rate
// of the fp32 MFMA, six of them run 2.7 times as fast. F16 weights need two parts (11 bits; five
// products). A Q3_K weight is d (one per super-block) times the integer scale * code, at most 128
// in magnitude and so exact in one bf16: three products, d applied to the super-block's sum.
//
// Rounding order. The w0 x0 products of 256 elements add up in an accumulator of their own
// that then goes into the output sum, and the other products, 2^-8 as large, in another: 16
// rounded additions per chunk and one per chunk, against one long chain of all.
//
// Tiling. A workgroup of WN x WK waves owns 32 WN weight rows x 32 MT tokens; wave (wn, wk)
// takes 32 rows and every WK-th chunk of 256 elements, and the WK partial sums of a row group
// are added through LDS in wk order at the end. In a chunk the MFMA's two lane halves h hold
// elements 128 h .. 128 h + 127, 32 of each per stage, so that a lane decodes whole 32-element
// units of its own row with the GEMV's decoders, and a lane's quarter super-blocks share one
// load of the raw bytes. The token side is split once per workgroup on its way into LDS
// (16-byte chunks swizzled by token: a wave's fragment reads spread over all banks), two
// stages of 64 WK elements in turn.
//
// Small values. The matrix cores take bf16 values below 2^-126 for zero, which the lower parts of
// fp32 values below 2^-101 are (1.1e-6 off at 2^-115, 3.6e-2 at 2^-130). So the activations, and fp32
// weights, are split times 2^26, and the sums go back by as much: exact, at any size. (The other
// types' weights have binary16 scales, 2^-24 and up.)
//
// Non-finite values. inf * 0 appears among the split products where fp32 would have inf, and a
// finite value that is above the largest bf16 times 2^26 rounds to inf. Any such input makes its outputs
// non-finite, so a wave's tile (32 rows x 32 tokens) that holds an output that is not finite is
// computed again on fp32 MFMA, and such outputs take its value. MI355X, us, all finite / one NaN
// token / all NaN / GEMV: Q3_K 4096 x 4096 at 301 rows 75 / 199 / 326 / 450, F32 at 64 39 / 168 /
// 166 / 187, Q8_1 at 32 31 / 139 / 138 / 57 (one lane per output, its dot product in series: Q3_K
// 4100 / 5500).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "float_units.h"
#include "ggml_blocks.h"
#include "launch.h"
#include "mfma_common.h"

namespace cllm_hip {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Parts of a weight: fp32 values 3, binary16 2, Q3_K's integers 1.
template <uint32_t T>
constexpr int wparts() { return T == T_F16 ? 2 : T == T_Q3_K ? 1 : 3; }

// The raw bytes a lane keeps for the four units 4 h + j (j = 0..3) of a chunk, and the values
// of unit j. Types of 32-element units load each unit when its stage comes; the super-block
// types load a half super-block once.
template <uint32_t T>
struct GUnit {
    static constexpr bool HALF = false;
    using Raw = typename FUnit<T>::Raw;
    __device__ __forceinline__ static Raw load(const uint8_t* row, int u) { return FUnit<T>::load(row, u); }
    __device__ __forceinline__ static void decode(const Raw& r, int u, float (&w)[32]) { FUnit<T>::decode(r, u, w); }
};
template <> struct GUnit<T_Q2_K> {
    static constexpr bool HALF = true;
    struct Raw { u32x4_a4 q0, q1; u32x2_a4 sc; uint32_t dd; };
    __device__ __forceinline__ static Raw load(const uint8_t* row, int u) {
        const uint8_t* blk = row + (size_t)(u >> 3) * 84;
        const int h = (u & 7) >> 2;
        Raw r;
        r.q0 = *(const u32x4_a4*)(blk + 16 + 32 * h);
        r.q1 = *(const u32x4_a4*)(blk + 32 + 32 * h);
        r.sc = *(const u32x2_a4*)(blk + 8 * h);
        r.dd = *(const uint32_t*)(blk + 80);
        return r;
    }
    __device__ __forceinline__ static void decode(const Raw& r, int u, float (&w)[32]) {
        const int j = u & 3;
        FUnit<T_Q2_K>::Raw v;
        v.q0 = r.q0;
        v.q1 = r.q1;
        v.sc = ((j & 2 ? r.sc.y : r.sc.x) >> (16 * (j & 1))) & 0xFFFFu;
        v.dd = r.dd;
        FUnit<T_Q2_K>::decode(v, u, w);
    }
};
template <> struct GUnit<T_Q3_K> {
    static constexpr bool HALF = true;
    using Raw = FUnit<T_Q3_K>::Raw;
    __device__ __forceinline__ static Raw load(const uint8_t* row, int u) { return FUnit<T_Q3_K>::load(row, u); }
    // the integers scale * code, d left out: fma(byte, scale, -4 scale) on bytes of code + 4
    __device__ __forceinline__ static void decode(const Raw& r, int u, float (&w)[32]) {
        const int h = (u & 7) >> 2, j = u & 3;
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            const float sc = (float)FUnit<T_Q3_K>::scale(r.sc, 8 * h + 2 * j + g), off = -4.0f * sc;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t q2 = (r.q[4 * g + i] >> (2 * j)) & 0x03030303u;
                uint32_t qv = q2 | (((r.hm[4 * g + i] >> (4 * h + j)) & 0x01010101u) << 2);
                asm volatile("" : "+v"(qv));  // keep the byte conversions (see codes16)
#pragma unroll
                for (int b = 0; b < 4; ++b) w[16 * g + 4 * i + b] = __builtin_fmaf(ubyte_f(qv, b), sc, off);
            }
        }
    }
};

constexpr float kUp = 0x1p26f;  // what operands are multiplied with before they are split

template <uint32_t T, int WN, int WK, int MT>
struct CfgF {
    static constexpr int THREADS = 64 * WN * WK;
    static constexpr int BN = 32 * WN, BM = 32 * MT;
    static constexpr int TASKS = BM * 8 / (64 * WN);      // 8-element pieces per thread and stage
    static constexpr int PART = BM * 128;                 // LDS bytes of one part of one K slice
    static constexpr int SLICE = 3 * PART;
    static constexpr int STAGE = WK * SLICE;
    static constexpr int RED = (WK - 1) * WN * MT * 16 * 64 * 4;  // the K parts' sums, at the end
    static constexpr int LDS = 2 * STAGE > RED ? 2 * STAGE : RED;
    static_assert(LDS <= 160 * 1024, "LDS budget");
    static_assert(TASKS * 64 * WN == BM * 8, "whole staging passes");
};

// A 32 x 32 tile in fp32 (v_mfma_f32_32x32x2f32), for the outputs that the split products could not
// represent: lane (h, r32) decodes unit 2 i + h of weight row wrow and reads the same unit of token
// row xr, and each pair of elements is one MFMA; 32 elements add up from zero before they join the
// tile (one chain over 1024 was 5.6e-7 off the 64-bit sums, this 1.5e-7, the GEMV 1.2e-7). Rows and
// tokens mix in no output, so the others' infinities stay theirs.
template <uint32_t T>
__device__ __forceinline__ wf16 tile_f32(const uint8_t* wrow, int units, const float* xr, int h) {
    wf16 s;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = 0.0f;
    typename FUnit<T>::Raw raw = FUnit<T>::load(wrow, min(h, units - 1));
    f32x4 xv[8];
    auto load_x = [&](int u) {
#pragma unroll
        for (int e = 0; e < 8; ++e) xv[e] = *(const f32x4*)(xr + 32 * u + 4 * e);
    };
    load_x(min(h, units - 1));
#pragma unroll 1
    for (int u0 = 0; u0 < units; u0 += 2) {
        const bool in = u0 + h < units;
        const int next = min(u0 + 2 + h, units - 1);
        float v[32], xe[32];
        FUnit<T>::decode(raw, min(u0 + h, units - 1), v);
#pragma unroll
        for (int e = 0; e < 32; ++e) {
            v[e] = in ? v[e] : 0.0f;
            xe[e] = in ? xv[e / 4][e % 4] : 0.0f;
        }
        raw = FUnit<T>::load(wrow, next);  // beside the MFMAs
        load_x(next);
#pragma unroll
        for (int e = 0; e < 32; e += 16) {
            wf16 c = {};
#pragma unroll
            for (int i = 0; i < 16; ++i) c = __builtin_amdgcn_mfma_f32_32x32x2f32(v[e + i], xe[e + i], c, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] += c[r];
        }
    }
    return s;
}

template <uint32_t T, int WN, int WK, int MT>
__global__ __launch_bounds__(64 * WN * WK) void k_gemm_f(const uint8_t* __restrict__ w,
                                                         size_t row_bytes, int k, int n, int m,
                                                         const float* __restrict__ x,
                                                         const float* __restrict__ bias,
                                                         float* __restrict__ y) {
    using C = CfgF<T, WN, WK, MT>;
    constexpr int PW = wparts<T>();
    constexpr float kDown = T == T_F32 ? 1.0f / kUp / kUp : 1.0f / kUp;
    extern __shared__ __align__(16) uint8_t lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wn = wave % WN, wk = wave / WN;
    const int h = lane >> 5, r32 = lane & 31;
    const int units = k / 32;

    // (weight block, token block), the token blocks of a weight block on one XCD (hardware
    // hands consecutive workgroups to the 8 XCDs in turn)
    const int mb = (m + C::BM - 1) / C::BM;
    const int g = gridDim.x, bid = blockIdx.x;
    const int lin = g % 8 == 0 ? (bid % 8) * (g / 8) + bid / 8 : bid;
    const int nblk = lin / mb, mblk = lin - nblk * mb;
    const int n0 = nblk * C::BN + wn * 32, m0 = mblk * C::BM;
    // rows and tokens past the matrix repeat the last one (their results are dropped)
    const uint8_t* wrow = w + (size_t)min(n0 + r32, n - 1) * row_bytes;

    // stage s: quarter j = s & 3 of chunk (s >> 2) WK + wk, one chunk per wave and step
    const int chunks = (units + 7) / 8;
    const int stages = (chunks + WK - 1) / WK * 4;

    // this thread's pieces of a stage: 8 elements of one token and K slice
    const float* xp[C::TASKS];
    uint32_t xdst[C::TASKS];
    int xu[C::TASKS];  // the piece's unit in stage 0
#pragma unroll
    for (int i = 0; i < C::TASKS; ++i) {
        const int task = (int)threadIdx.x + i * C::THREADS;
        const int c = task & 7, t = (task >> 3) % C::BM, ks = (task >> 3) / C::BM;
        xu[i] = 8 * ks + 4 * (c >> 2);
        xp[i] = x + (size_t)min(m0 + t, m - 1) * k + 8 * (c & 3);
        xdst[i] = (uint32_t)(ks * C::SLICE + t * 128 + ((c ^ (t & 7)) << 4));
    }
    f32x4 xr[C::TASKS][2];
    auto load_x = [&](int s) {
#pragma unroll
        for (int i = 0; i < C::TASKS; ++i) {
            const int u = xu[i] + 8 * WK * (s >> 2) + (s & 3);
            const float* p = xp[i] + 32 * min(u, units - 1);
            xr[i][0] = *(const f32x4*)p;
            xr[i][1] = *(const f32x4*)(p + 4);
        }
    };
    auto store_x = [&](int s, uint8_t* st) {
#pragma unroll
        for (int i = 0; i < C::TASKS; ++i) {
            // zeros past K (times the token's last values: where those are infinite, so are its outputs)
            const float up = xu[i] + 8 * WK * (s >> 2) + (s & 3) < units ? kUp : 0.0f;
            const f32x4 lo4 = xr[i][0], hi4 = xr[i][1];
            float v[8] = {lo4.x, lo4.y, lo4.z, lo4.w, hi4.x, hi4.y, hi4.z, hi4.w};
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] *= up;
            wbf8 p[3];
            split8<3>(v, p);
#pragma unroll
            for (int q = 0; q < 3; ++q) *(wbf8*)(st + q * C::PART + xdst[i]) = p[q];
        }
    };

    wf16 hi[MT], lo[MT], acc[MT];
#pragma unroll
    for (int a = 0; a < MT; ++a)
#pragma unroll
        for (int r = 0; r < 16; ++r) hi[a][r] = lo[a][r] = acc[a][r] = 0.0f;

    auto unit_of = [&](int s) { return 8 * ((s >> 2) * WK + wk) + 4 * h + (s & 3); };
    typename GUnit<T>::Raw raw = GUnit<T>::load(wrow, min(unit_of(0), units - 1));
    // the weight operand of K step q (elements 8 q .. 8 q + 7 of the lane's unit) of stage j
    // (a clamped unit's values meet zeros of x)
    auto frag = [&](int j, int q, wbf8 (&a)[PW]) {
        float wv[32];
        GUnit<T>::decode(raw, GUnit<T>::HALF ? 4 * h + j : 0, wv);
        if constexpr (T == T_F32) {
#pragma unroll
            for (int e = 0; e < 8; ++e) wv[8 * q + e] *= kUp;
        }
        split8<PW>(wv + 8 * q, a);
    };
    wbf8 afr[2][PW];
    frag(0, 0, afr[0]);
    load_x(0);
    store_x(0, lds);
    __syncthreads();

    const uint8_t* bbase = lds + wk * C::SLICE + r32 * 128;
    // four stages (one chunk) per turn: j is a constant in each
    for (int s4 = 0; s4 < stages; s4 += 4) {
        float dsb = 1.0f;  // Q3_K: d of this lane's row and chunk
        if constexpr (T == T_Q3_K) dsb = f16_to_f32(raw.d);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int s = s4 + j;
            const uint8_t* cur = bbase + (j & 1) * C::STAGE;
            // the next stage's loads (past the last one clamped in bounds and not used)
            load_x(s + 1);
            typename GUnit<T>::Raw next;
            if (!GUnit<T>::HALF || j == 3) next = GUnit<T>::load(wrow, min(unit_of(s + 1), units - 1));
            // items i = K step * MT + token tile: the next item's fragments are read and the
            // next K step's weights decoded beside this one's MFMAs
            wbf8 b[2][3];
            auto read = [&](int i) {
                const uint8_t* p = cur + (i % MT) * (32 * 128) + (((4 * h + i / MT) ^ (r32 & 7)) << 4);
#pragma unroll
                for (int u = 0; u < 3; ++u) b[i & 1][u] = *(const wbf8*)(p + u * C::PART);
            };
            read(0);
#pragma unroll
            for (int i = 0; i < 4 * MT; ++i) {
                const int q = i / MT, a = i % MT;
                __builtin_amdgcn_sched_barrier(0);
                // two waves of the workgroup share a SIMD: the one behind in its stage gets it
                // (70.4 -> 67.8 us on Q3_K 4096 x 4096 at 301 rows)
                if (WN * WK > 4 && i == 0) __builtin_amdgcn_s_setprio(2);
                if (WN * WK > 4 && i == 2 * MT) __builtin_amdgcn_s_setprio(1);
                if (i + 1 < 4 * MT) read(i + 1);
                if (i % MT == 0) {
                    if (q == 3 && (!GUnit<T>::HALF || j == 3)) raw = next;
                    frag((j + (q == 3)) & 3, (q + 1) & 3, afr[(q + 1) & 1]);
                }
                const wbf8 (&w8)[PW] = afr[q & 1];
                const wbf8 (&x8)[3] = b[i & 1];
                hi[a] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w8[0], x8[0], hi[a], 0, 0, 0);
                lo[a] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w8[0], x8[2], lo[a], 0, 0, 0);
                if constexpr (PW > 2) lo[a] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w8[2], x8[0], lo[a], 0, 0, 0);
                if constexpr (PW > 1) lo[a] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w8[1], x8[1], lo[a], 0, 0, 0);
                lo[a] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w8[0], x8[1], lo[a], 0, 0, 0);
                if constexpr (PW > 1) lo[a] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w8[1], x8[0], lo[a], 0, 0, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);  // the next item's LDS reads
#pragma unroll
                for (int u = 0; u < (PW == 1 ? 3 : PW == 2 ? 5 : 6); ++u) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // an MFMA
                    __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);  // VALU beside it
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            if (WN * WK > 4) __builtin_amdgcn_s_setprio(0);
            store_x(s + 1, lds + ((j + 1) & 1) * C::STAGE);
            __syncthreads();
            // Q8_1: half chunks, and what rounding takes off goes to the small products' sum.
            // (The GEMV's sums of exact codes per block round less for this type than for the
            // others: 9.7e-8 to 1.1e-7 off the 64-bit result, 1.3e-7 here without this.)
            if constexpr (T == T_Q8_1) {
                if (j & 1) {
#pragma unroll
                    for (int a = 0; a < MT; ++a)
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            const float t = acc[a][r] + hi[a][r], v = t - acc[a][r];
                            lo[a][r] += (acc[a][r] - (t - v)) + (hi[a][r] - v);
                            acc[a][r] = t;
                            hi[a][r] = 0.0f;
                        }
                }
            }
        }
        if constexpr (T == T_Q8_1) continue;
        // the chunk's sums into the output's; for Q3_K times d of the lane's 16 output rows,
        // held by lanes 8 (r / 4) + 4 h + r % 4
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            if constexpr (T == T_Q3_K) {
                const float d = __shfl(dsb, 8 * (r >> 2) + 4 * h + (r & 3));
#pragma unroll
                for (int a = 0; a < MT; ++a) {
                    acc[a][r] = __builtin_fmaf(d, hi[a][r] + lo[a][r], acc[a][r]);
                    lo[a][r] = 0.0f;
                }
            } else {
#pragma unroll
                for (int a = 0; a < MT; ++a) acc[a][r] += hi[a][r];
            }
#pragma unroll
            for (int a = 0; a < MT; ++a) hi[a][r] = 0.0f;
        }
    }
#pragma unroll
    for (int a = 0; a < MT; ++a)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[a][r] += lo[a][r];

    // the WK partial sums of a row group, in wk order (the stage buffers are free: the last
    // stage ended with a barrier)
    if constexpr (WK > 1) {
        float* red = (float*)lds;
        if (wk > 0) {
#pragma unroll
            for (int a = 0; a < MT; ++a)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    red[((((wk - 1) * WN + wn) * MT + a) * 16 + r) * 64 + lane] = acc[a][r];
        }
        __syncthreads();
        if (wk > 0) return;
        for (int p = 0; p < WK - 1; ++p)
#pragma unroll
            for (int a = 0; a < MT; ++a)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    acc[a][r] += red[(((p * WN + wn) * MT + a) * 16 + r) * 64 + lane];
    }

    float bv[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) bv[r] = 0.0f;
    if (bias) {
#pragma unroll
        for (int r = 0; r < 16; ++r) bv[r] = bias[min(n0 + 8 * (r >> 2) + 4 * h + (r & 3), n - 1)];
    }
#pragma unroll
    for (int a = 0; a < MT; ++a) {
        const int t = m0 + 32 * a + r32;
        // (times kDown is exact, so one FMA rounds as the bias's addition does)
        auto store = [&](int r, float v, float down) {
            const int row = n0 + 8 * (r >> 2) + 4 * h + (r & 3);
            if (row < n) y[(size_t)t * n + row] = bias ? __builtin_fmaf(v, down, bv[r]) : v * down;
        };
        float nan = 0.0f;  // once an output is not finite
#pragma unroll
        for (int r = 0; r < 16; ++r) nan = __builtin_fmaf(acc[a][r], 0.0f, nan);
        if (__any(nan != 0.0f)) {
            const wf16 f = tile_f32<T>(wrow, units, x + (size_t)min(t, m - 1) * k, h);
            if (t >= m) continue;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const bool fin = fabsf(acc[a][r]) < INFINITY;
                store(r, fin ? acc[a][r] : f[r], fin ? kDown : 1.0f);
            }
            continue;
        }
        if (t >= m) continue;
#pragma unroll
        for (int r = 0; r < 16; ++r) store(r, acc[a][r], kDown);
    }
}

template <uint32_t T, int WN, int WK, int MT>
hipError_t launch_cfg(const uint8_t* w, int k, int n, int m, const float* x, const float* bias,
                      float* y, hipStream_t stream) {
    using C = CfgF<T, WN, WK, MT>;
    static LdsLimit limit;
    const hipError_t e = limit.raise((const void*)k_gemm_f<T, WN, WK, MT>, C::LDS);
    if (e != hipSuccess) return e;
    const size_t row_bytes = (size_t)(k / block_elems(T)) * block_bytes(T);
    const unsigned grid = (unsigned)(((n + C::BN - 1) / C::BN) * ((m + C::BM - 1) / C::BM));
    hipLaunchKernelGGL((k_gemm_f<T, WN, WK, MT>), dim3(grid), dim3(C::THREADS), C::LDS, stream, w,
                       row_bytes, k, n, m, x, bias, y);
    return hipGetLastError();
}

template <uint32_t T>
hipError_t launch_t(int shape, const uint8_t* w, int k, int n, int m, const float* x,
                    const float* bias, float* y, hipStream_t stream) {
    switch (shape) {
        case 1: return launch_cfg<T, 4, 2, 2>(w, k, n, m, x, bias, y, stream);
        case 2: return launch_cfg<T, 2, 2, 1>(w, k, n, m, x, bias, y, stream);
        default: return launch_cfg<T, 1, 4, 1>(w, k, n, m, x, bias, y, stream);
    }
}

int cus() {
    static const int n = [] {
        int dev = 0, c = 0;
        return hipGetDevice(&dev) == hipSuccess &&
                       hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && c > 0
                   ? c
                   : 256;
    }();
    return n;
}

// The tile shape for a batch (1: 128 x 64, K on 2 waves; 2: 64 x 32, K on 2; 3: 32 x 32, K on
// 4), or 0 where the GEMV is faster, by the time each would take. A stage (64 WK elements)
// takes a workgroup about the same time however many run beside it, up to one per CU; two or
// three of shape 2 share a CU. The constants fit the measurements below and their like; a shape
// has to beat the GEMV by 3 us of that estimate. MI355X, cold weights, us (GEMV / shapes 1 / 2 / 3):
//   Q3_K 4096 x 4096,  16 rows:  26.7 /  66 /  37 /  28     F32 4096 x 4096, 301 rows:  810 / 94 / 124 / 167
//                      32:       55.5 /  66 /  38 /  29     Q4_1 4096 x 4096, 301:      476 / 85 /  93 / 142
//                      64:        100 /  66 /  38 /  30     Q2_K 14336 x 4096, 16:       73 / 86 /  42 /  56
//                     128:        206 /  66 /  39 /  55                        64:      253 / 87 /  66 / 108
//                     301:        447 /  67 /  73 / 131     Q4_1 300 x 2048, 64:         11 / 45 /  23 /  17
//                                                                          200:         22 / 45 /  25 /  19
int shape_for(uint32_t type, int k, int n, int m) {
    if (m < 8) return 0;  // short batches run the GEMV's code, row for row
    const int c = cus(), chunks = (k + 255) / 256;
    const float f = type == T_F32 ? 1.4f : type == T_F16 ? 1.1f : type == T_Q3_K ? 1.0f : 1.3f;
    auto rounds = [&](int bn, int bm) {
        const int64_t wgs = (int64_t)((n + bn - 1) / bn) * ((m + bm - 1) / bm);
        return (float)((wgs + c - 1) / c);
    };
    const float st2 = 4.0f * (float)((chunks + 1) / 2), st4 = 4.0f * (float)((chunks + 3) / 4);
    const float us[3] = {f * st2 * 2.0f * rounds(128, 64), f * st2 * (0.55f + 0.55f * rounds(64, 32)),
                         f * st4 * 1.65f * rounds(32, 32)};
    const int best = us[0] <= us[1] && us[0] <= us[2] ? 0 : us[1] <= us[2] ? 1 : 2;
    const float gemv = 4.0f + (float)m * (float)n * (float)k * (type == T_F32 ? 1.6e-7f : 0.9e-7f);
    return us[best] + 3.0f < gemv ? best + 1 : 0;
}

int shape_of(uint32_t type, int k, int n, int m) {
    if (k % 32 != 0 || !gemv_f_supported(type)) return 0;
    const int knob = tuning().gemm_f.load(std::memory_order_relaxed);
    if (knob == 9) return 0;
    if (knob != 0) return m >= 2 ? knob : 0;
    return shape_for(type, k, n, m);
}

}  // namespace

bool gemm_f_takes(uint32_t type, int k, int n, int m) { return shape_of(type, k, n, m) != 0; }

hipError_t launch_gemm_f(uint32_t type, const uint8_t* w, int k, int n, int m, const float* x,
                         const float* bias, float* y, hipStream_t stream) {
    const int shape = shape_of(type, k, n, m);
    if (shape == 0) return hipErrorNotSupported;
    switch (type) {
        case T_F32: return launch_t<T_F32>(shape, w, k, n, m, x, bias, y, stream);
        case T_F16: return launch_t<T_F16>(shape, w, k, n, m, x, bias, y, stream);
        case T_Q4_1: return launch_t<T_Q4_1>(shape, w, k, n, m, x, bias, y, stream);
        case T_Q5_1: return launch_t<T_Q5_1>(shape, w, k, n, m, x, bias, y, stream);
        case T_Q8_1: return launch_t<T_Q8_1>(shape, w, k, n, m, x, bias, y, stream);
        case T_Q2_K: return launch_t<T_Q2_K>(shape, w, k, n, m, x, bias, y, stream);
        case T_Q3_K: return launch_t<T_Q3_K>(shape, w, k, n, m, x, bias, y, stream);
        default: return hipErrorNotSupported;
    }
}

}  // namespace cllm_hip
