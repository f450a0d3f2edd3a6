// k_attention.hip -- the float ops between the linear layers on the device: NEOX RoPE and
// grouped-query attention over a KV cache (decode and prefill).
//
// Reference (src/core/engine.cpp):
//   apply_rope (41-56): per head, pairs (i, i + half), theta = pos / base^(i / half),
//     x_i' = x_i cos - x_{i+half} sin, x_{i+half}' = x_i sin + x_{i+half} cos;
//   attention (114-146): per query head h (KV head h / n_rep), s_t = dot(q_h, k_t) / sqrt(d)
//     over the t < seq cached positions, softmax (max subtracted, exp, sum), then
//     out_h = sum_t (e_t / sum) v_t; decode (495) and prefill (581-583, query t of the
//     batch sees pos0 + t + 1 positions).
//
// Three attention kernels: k_attention (below; decode, and a few rows over a long cache),
// k_attention_mfma (many query rows: at head_dim 64 and 128 on bf16 MFMA with fp32 operands split
// in three, at 256 on fp32 MFMA) and k_attention_mfma_f32 (many query rows at head_dim 64 and 128
// over caches of 4 GiB and more, on fp32 MFMA); the layouts of the latter two are described above
// them.
//
// Attention layout. One workgroup per (KV head, query row, sequence split); it serves the
// n_rep query heads of that KV head, so every K and V row is loaded once for all of them. Its
// waves walk the positions on their own (the layout is described at the kernel); the softmax is
// online (running max and sum, the partial output rescaled when the max grows).
// Long sequences are split over several workgroups whose (max, sum, unnormalised output)
// partials the last of them to finish combines (a per-(row, KV head) arrival counter), so a
// decode step (one query row) still spreads over the device in one launch. The summation
// order differs from the reference's (per-chunk and per-split partial sums, output divided
// by the sum once); the arithmetic is otherwise the same
// fp32 operations with the device's expf, sinf, cosf and powf.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "device_utils.h"
#include "launch.h"
#include "mfma_common.h"

namespace cllm_hip {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------------- RoPE

// grid (rows, groups of kRopeHeads heads): row t has position pos0 + t; heads past n_heads belong
// to the second tensor x2 (the keys), so the queries and keys of a layer turn in one launch. The
// head_dim / 2 angles of the row are formed once per workgroup (a power, a cosine and a sine each)
// and turn all of its heads: with a workgroup per head that arithmetic, on a quarter of the lanes,
// took 11.8 us for 512 rows of 32 + 8 heads of 128; now 6.2 (20 MB moved). From ten heads on the
// angles no longer show there (2 / 4 / 10 / 20 heads per workgroup, a call every 10.7 / 8.0 / 7.5 /
// 7.4 us); 2048 rows take 34 / 24 / 17.7 / 15.6.
constexpr int kRopeHeads = 10;
__global__ __launch_bounds__(256) void k_rope_neox(float* __restrict__ x, int n_heads,
                                                   float* __restrict__ x2, int n_heads2,
                                                   int head_dim, int pos0, float base) {
    __shared__ float cs[2][256];
    const int t = blockIdx.x;
    const int half = head_dim / 2;
    if ((int)threadIdx.x < half) {
        const int i = threadIdx.x;
        const float theta = __fdiv_rn((float)(pos0 + t), powf(base, __fdiv_rn((float)i, (float)half)));
        cs[0][i] = cosf(theta);
        cs[1][i] = sinf(theta);
    }
    __syncthreads();
    const int h0 = blockIdx.y * kRopeHeads, heads = min(kRopeHeads, n_heads + n_heads2 - h0);
    for (int p = threadIdx.x; p < heads * half; p += 256) {
        const int hh = p / half, i = p - hh * half, h = h0 + hh;
        float* xh = h >= n_heads ? x2 + ((size_t)t * n_heads2 + (h - n_heads)) * head_dim
                                 : x + ((size_t)t * n_heads + h) * head_dim;
        const float c = cs[0][i], s = cs[1][i];
        const float x0 = xh[i], x1 = xh[i + half];
        xh[i] = __builtin_fmaf(x0, c, -__fmul_rn(x1, s));
        xh[i + half] = __builtin_fmaf(x0, s, __fmul_rn(x1, c));
    }
}

// ----------------------------------------------------------------------------- attention

constexpr int kThreads = 256;
constexpr int kChunk = 64;       // a sequence split is a multiple of this many positions
constexpr int kLanesPerPos = 16; // lanes sharing one K row
constexpr int kMaxRep = 8;       // query heads per KV head
constexpr int kAttnCounters = 1024;  // (row, KV head) pairs a split launch may have
constexpr int kMaxSplits = 256;      // sequence splits per (row, KV head)

// HD = head_dim (multiple of 64, at most 256). Partials of split z for query head hq of row
// t: part[((t * n_head + hq) * S + z) * (HD + 4) + ...] = unnormalised output [HD], max, sum
// (two floats of padding keep every row 16-byte aligned for the combine's vector loads).
// With one split, the normalised output goes straight to out.
//
// Waves work alone: no barrier and no LDS between the query's staging and the end. A wave
// takes 4 P positions at a time, P in each of its four 16-lane rows; lane seg of a row holds
// dims 64 i + 4 seg .. + 3 (i < HD / 64) of the K row, the V row, every query head of the group
// and every head's output (a load instruction reads 256 contiguous bytes of four cache rows).
// The P NREP scores of a row's positions are reduced together: each DPP step halves the number
// of values a lane still carries, so lane idx(j, r) ends with the score of position j and head
// r, takes its exponential once, and hands it to the row by a DPP broadcast. Maxima and sums
// are per row of lanes (and head); the 16 rows of the workgroup meet at the end.
//
// What bounds it: the cache stream. One chunk of 64 positions per step with three barriers and
// a reduction per (position, head) took 54 us over 8192 positions of 8 KV heads (67 MB) and
// 15 us over 1024; this form takes 23 and 11.5, of which 9 go to the launch, the rotation and
// the meeting of the splits (MI355X, 32 query heads of 128).
//
// (Nontemporal loads of the cache rows measured slower: 31.7 against 24.8 us at 8192.)
//
// rope_base > 0 (one query row, a decode step): the queries and the key row at pos0 arrive
// unrotated and the kernel applies the NEOX rotation of k_rope_neox itself, to the queries in
// registers and to the key row as it loads it, writing the rotated key row back to k_new (the
// cache row pos0, read by no other workgroup: only the split holding pos0 covers it; waves of
// this workgroup that clamp to it mask its score). k_new points into the key cache, so kc
// carries no __restrict__: the compiler may not treat the cache as unwritten by this kernel.
template <int CTRL>
__device__ __forceinline__ float row_bcast(float v) { return dpp_f32<0x150 + CTRL>(v); }
// the value of lane LANE of each 16-lane row (LANE constant after unrolling)
__device__ __forceinline__ float bcast16(float v, int lane) {
    switch (lane) {
        case 0: return row_bcast<0>(v);
        case 1: return row_bcast<1>(v);
        case 2: return row_bcast<2>(v);
        case 3: return row_bcast<3>(v);
        case 4: return row_bcast<4>(v);
        case 5: return row_bcast<5>(v);
        case 6: return row_bcast<6>(v);
        case 7: return row_bcast<7>(v);
        case 8: return row_bcast<8>(v);
        case 9: return row_bcast<9>(v);
        case 10: return row_bcast<10>(v);
        case 11: return row_bcast<11>(v);
        case 12: return row_bcast<12>(v);
        case 13: return row_bcast<13>(v);
        case 14: return row_bcast<14>(v);
        default: return row_bcast<15>(v);
    }
}

// One step of the joint reduction over a 16-lane row: lanes whose bit is clear keep the first
// half of the values, the others the second, each plus the partner's.
template <int CTRL, int V>
__device__ __forceinline__ void halve(float (&v)[V], int n, bool upper) {
#pragma unroll
    for (int i = 0; i < V / 2; ++i) {
        if (i >= n / 2) break;
        const float keep = upper ? v[i + n / 2] : v[i], give = upper ? v[i] : v[i + n / 2];
        v[i] = keep + dpp_f32<CTRL>(give);
    }
}

// Positions per lane row and step: as many as leave registers for two waves per SIMD (one at
// head_dim 256 with 8 heads), at most 16 scores.
template <int HD, int NREP>
constexpr int attention_p() { return HD == 256 ? (NREP == 8 ? 1 : NREP == 4 ? 2 : 4) : NREP == 8 ? 2 : 4; }

template <int HD, int NREP>
__global__ __launch_bounds__(kThreads, HD == 256 && NREP == 8 ? 1 : 2) void k_attention(
    const float* __restrict__ q, const float* kc, const float* __restrict__ vc,
    int n_head, int n_kv, int pos0, int split_len, float scale, float* __restrict__ part,
    int* __restrict__ counters, float* __restrict__ out, float rope_base, float* k_new) {
    constexpr int PER = HD / kLanesPerPos;   // dims per lane (4, 8 or 16)
    constexpr int NB = PER / 4;              // 16-byte pieces per lane and row
    constexpr int P = attention_p<HD, NREP>();  // positions per lane row and step
    constexpr int V = P * NREP;              // scores per lane row and step (4, 8 or 16)
    constexpr int DUP = 16 / V;              // lanes that end with the same score
    constexpr int STEP = 4 * P;
    constexpr int W = kThreads / 64;

    const int kvh = blockIdx.x, t = blockIdx.y, z = blockIdx.z, S = gridDim.z;
    const int n_rep = n_head / n_kv;
    const int kv_dim = n_kv * HD;
    const int L = pos0 + t + 1;
    const int begin = z * split_len;
    const int end = min(L, begin + split_len);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int seg = lane & 15, sub = lane >> 4;

    const float* kg = kc + (size_t)kvh * HD + 4 * seg;
    const float* vg = vc + (size_t)kvh * HD + 4 * seg;
    float kf[P][PER], vf[P][PER];
    // position c0 + 4 j + sub, clamped to the split's last (its score is then masked)
    auto load = [&](float (&x)[P][PER], const float* base, int c0) {
#pragma unroll
        for (int j = 0; j < P; ++j) {
            const float* row = base + (size_t)min(c0 + 4 * j + sub, end - 1) * kv_dim;
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const f32x4 v = *(const f32x4*)(row + 64 * i);
                x[j][4 * i] = v.x; x[j][4 * i + 1] = v.y; x[j][4 * i + 2] = v.z; x[j][4 * i + 3] = v.w;
            }
        }
    };
    float qv[NREP][PER];
#pragma unroll
    for (int r = 0; r < NREP; ++r) {
        const float* qh = q + ((size_t)t * n_head + kvh * n_rep + min(r, n_rep - 1)) * HD + 4 * seg;
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const f32x4 v = *(const f32x4*)(qh + 64 * i);
            qv[r][4 * i] = v.x; qv[r][4 * i + 1] = v.y; qv[r][4 * i + 2] = v.z; qv[r][4 * i + 3] = v.w;
        }
    }
    // (after the queries: loads return in order, and the queries are rotated first)
    int c0 = begin + wave * STEP;
    load(kf, kg, c0);
    load(vf, vg, c0);
    // NEOX rotation at position pos0: dim i pairs with i + HD / 2, held by the same lane (HD >=
    // 128) or by lane seg ^ 8 (HD = 64). The angles of the pairs, one per thread, go through LDS.
    const bool rope = rope_base > 0.0f;
    __shared__ float rope_cs[2][HD / 2];
    float rc[PER], rs[PER];
    auto rotate = [&](float (&x)[PER]) {
        float o[PER];
#pragma unroll
        for (int e = 0; e < PER; ++e) {
            const bool lo = HD == 64 ? seg < 8 : e < PER / 2;
            const float other = HD == 64 ? dpp_f32<0x128>(x[e]) : x[(e + PER / 2) % PER];  // row_ror:8
            const float x0 = lo ? x[e] : other, x1 = lo ? other : x[e];
            o[e] = lo ? __builtin_fmaf(x0, rc[e], -__fmul_rn(x1, rs[e]))
                      : __builtin_fmaf(x0, rs[e], __fmul_rn(x1, rc[e]));
        }
#pragma unroll
        for (int e = 0; e < PER; ++e) x[e] = o[e];
    };
    if (rope) {
        if (threadIdx.x < HD / 2) {
            const int i = threadIdx.x;
            const float theta = __fdiv_rn((float)pos0, powf(rope_base, __fdiv_rn((float)i, (float)(HD / 2))));
            rope_cs[0][i] = cosf(theta);
            rope_cs[1][i] = sinf(theta);
        }
        // a barrier that orders LDS only: the cache rows stay in flight
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
#pragma unroll
        for (int e = 0; e < PER; ++e) {
            const int d = (64 * (e >> 2) + 4 * seg + (e & 3)) % (HD / 2);
            rc[e] = rope_cs[0][d];
            rs[e] = rope_cs[1][d];
        }
#pragma unroll
        for (int r = 0; r < NREP; ++r) rotate(qv[r]);
    }

    float acc[NREP][PER];
#pragma unroll
    for (int r = 0; r < NREP; ++r)
#pragma unroll
        for (int e = 0; e < PER; ++e) acc[r][e] = 0.0f;
    // running maximum and sum of this lane's head (lanes with the same head agree)
    float m_run = -INFINITY, l_run = 0.0f;
    const int my_j = seg / DUP / NREP;  // the position of a step whose score this lane ends with

    for (; c0 < end; c0 += W * STEP) {
        if (rope && c0 <= pos0 && pos0 < c0 + STEP) {  // the new key row
#pragma unroll
            for (int j = 0; j < P; ++j) {
                float rot[PER];
#pragma unroll
                for (int e = 0; e < PER; ++e) rot[e] = kf[j][e];
                rotate(rot);
                if (c0 + 4 * j + sub == pos0) {
                    float* kw = k_new + kvh * HD + 4 * seg;
#pragma unroll
                    for (int i = 0; i < NB; ++i) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) kf[j][4 * i + e] = rot[4 * i + e];
                        *(f32x4*)(kw + 64 * i) = f32x4{rot[4 * i], rot[4 * i + 1], rot[4 * i + 2], rot[4 * i + 3]};
                    }
                }
            }
        }
        float s[V];
#pragma unroll
        for (int j = 0; j < P; ++j)
#pragma unroll
            for (int r = 0; r < NREP; ++r) {
                float d = 0.0f;
#pragma unroll
                for (int e = 0; e < PER; ++e) d = __builtin_fmaf(qv[r][e], kf[j][e], d);
                s[j * NREP + r] = d;
            }
        // (loads of the next step, past the split's last one clamped in bounds and not used)
        load(kf, kg, min(c0 + W * STEP, end - 1));
        // lanes seg ^ 8, seg ^ 7 (a half row's mirror), seg ^ 2, seg ^ 1: together the 16 lanes
        halve<0x128, V>(s, V, seg & 8);
        halve<DPP_ROW_HALF_MIRROR, V>(s, V / 2, seg & 4);
        if constexpr (V >= 8) halve<DPP_QUAD_SWAP2, V>(s, V / 4, seg & 2);
        else s[0] += dpp_f32<DPP_QUAD_SWAP2>(s[0]);
        if constexpr (V >= 16) halve<DPP_QUAD_SWAP1, V>(s, V / 8, seg & 1);
        else s[0] += dpp_f32<DPP_QUAD_SWAP1>(s[0]);
        const float sv = c0 + 4 * my_j + sub < end ? __fmul_rn(s[0], scale) : -INFINITY;
        // the same head's lanes: seg ^ 8 (two positions) and seg ^ 4 (four)
        float mx = sv;
        if constexpr (P >= 2) mx = fmaxf(mx, dpp_f32<0x128>(mx));
        if constexpr (P == 4) mx = fmaxf(mx, dpp_f32<0x1B>(dpp_f32<DPP_ROW_HALF_MIRROR>(mx)));
        const float mn = fmaxf(m_run, mx);
        const float pr = sv == -INFINITY ? 0.0f : expf(sv - mn);
        const float cr = m_run == -INFINITY ? 0.0f : expf(m_run - mn);
        float ps = pr;
        if constexpr (P >= 2) ps += dpp_f32<0x128>(ps);
        if constexpr (P == 4) ps += dpp_f32<0x1B>(dpp_f32<DPP_ROW_HALF_MIRROR>(ps));
        m_run = mn;
        l_run = __builtin_fmaf(l_run, cr, ps);
#pragma unroll
        for (int r = 0; r < NREP; ++r) {
            const float c = bcast16(cr, r * DUP);
#pragma unroll
            for (int e = 0; e < PER; ++e) acc[r][e] *= c;
        }
#pragma unroll
        for (int j = 0; j < P; ++j)
#pragma unroll
            for (int r = 0; r < NREP; ++r) {
                const float p = bcast16(pr, (j * NREP + r) * DUP);
#pragma unroll
                for (int e = 0; e < PER; ++e) acc[r][e] = __builtin_fmaf(p, vf[j][e], acc[r][e]);
            }
        load(vf, vg, min(c0 + W * STEP, end - 1));
    }

    // The 16 lane rows' partials: maxima and sums through LDS, each row's output scaled to the
    // common maximum, the four rows of a wave added across its lanes, the four waves through LDS.
    __shared__ float wpart[W][NREP * HD];
    __shared__ float mrow[4 * W][NREP], lrow[4 * W][NREP], m_all[NREP], l_all[NREP];
    if (seg < NREP * DUP && seg % DUP == 0) {
        mrow[wave * 4 + sub][seg / DUP] = m_run;
        lrow[wave * 4 + sub][seg / DUP] = l_run;
    }
    __syncthreads();
    if (threadIdx.x < NREP) {
        const int r = threadIdx.x;
        float M = -INFINITY, l = 0.0f;
#pragma unroll
        for (int i = 0; i < 4 * W; ++i) M = fmaxf(M, mrow[i][r]);
#pragma unroll
        for (int i = 0; i < 4 * W; ++i) {
            const float m = mrow[i][r], e = expf(m - M);
            const float w = m == -INFINITY ? 0.0f : e;
            l = __builtin_fmaf(w, lrow[i][r], l);
            mrow[i][r] = w;
        }
        m_all[r] = M;
        l_all[r] = l;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < NREP; ++r) {
        if (r >= n_rep) break;
        const float w = mrow[wave * 4 + sub][r];
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            float o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                o[e] = acc[r][4 * i + e] * w;
                o[e] += __shfl_xor(o[e], 16, 64);
                o[e] += __shfl_xor(o[e], 32, 64);
            }
            if (sub == 0) *(f32x4*)&wpart[wave][r * HD + 64 * i + 4 * seg] = f32x4{o[0], o[1], o[2], o[3]};
        }
    }
    __syncthreads();
    if (S == 1) {
        for (int o = threadIdx.x; o < n_rep * HD; o += kThreads) {
            const int r = o / HD, d = o - r * HD;
            const float v = (wpart[0][o] + wpart[1][o]) + (wpart[2][o] + wpart[3][o]);
            out[((size_t)t * n_head + kvh * n_rep + r) * HD + d] = __fdiv_rn(v, l_all[r]);
        }
        return;
    }
    // Several splits: write this split's partial; the last split of (row, KV head) to
    // arrive, found by a counter it resets, combines them all. The partials cross XCDs, whose
    // L2s are not coherent with each other, so they are stored and loaded as relaxed
    // agent-scope atomics (coherent device-wide by themselves; no L2-wide fence).
    for (int o = threadIdx.x; o < n_rep * HD; o += kThreads) {
        const int r = o / HD, d = o - r * HD;
        const float v = (wpart[0][o] + wpart[1][o]) + (wpart[2][o] + wpart[3][o]);
        float* pp = part + (((size_t)t * n_head + kvh * n_rep + r) * S + z) * (HD + 4);
        __hip_atomic_store(pp + d, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (d == 0) {
            __hip_atomic_store(pp + HD, m_all[r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(pp + HD + 1, l_all[r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    __builtin_amdgcn_s_waitcnt(0);  // this thread's partial stores have completed
    __syncthreads();
    __shared__ int last;
    if (threadIdx.x == 0) {
        int* cnt = counters + (size_t)t * n_kv + kvh;
        const int arrived = __hip_atomic_fetch_add(cnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        last = arrived == S - 1;
        if (arrived == S - 1) __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!last) return;
    // out = sum_z e^(m_z - M) o_z / sum_z e^(m_z - M) l_z, per head of the group.
    //
    // Each thread takes four consecutive dims of one head over one of G ranges of the splits
    // and reads them as one 16-byte load per split: a buffer load with the SC1 bit, the same
    // device-scope cache policy as the agent-scope atomic loads below, over this (row, KV
    // head)'s partial rows. Sixteen splits at a time are in flight, the first sixteen beside the
    // maxima and sums; the ranges are added through LDS in order (the wave partials are consumed).
    typedef float f32x4v __attribute__((ext_vector_type(4)));
    const float* pg = part + ((size_t)t * n_head + kvh * n_rep) * S * (HD + 4);
    const __amdgpu_buffer_rsrc_t prs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)pg, (short)0, (int)((size_t)n_rep * S * (HD + 4) * sizeof(float)), 0x00020000);
    constexpr int Q = HD / 4;
    const int outs = n_rep * Q;
    const int G = outs <= kThreads / 4 ? 4 : outs <= kThreads / 2 ? 2 : 1;
    const int zlen = (S + G - 1) / G;
    auto ld16 = [&](int o, int zz, uint32_t lead, f32x4v (&v)[16]) {  // (offsets past the rows read as zero)
        const int gi = o / outs, oo = o - gi * outs;
        const int r = oo / Q, d = 4 * (oo - r * Q), z1 = min(S, (gi + 1) * zlen);
        const uint32_t off = (uint32_t)(((r * S + gi * zlen + zz) * (HD + 4) + d) * sizeof(float)) + lead;
#pragma unroll
        for (int u = 0; u < 16; ++u)
            v[u] = __builtin_bit_cast(f32x4v, __builtin_amdgcn_raw_buffer_load_b128(
                prs, gi * zlen + zz + u < z1 ? off + u * (uint32_t)((HD + 4) * sizeof(float)) : 0x7FFFFFF0u, 0, 16));
    };
    uint32_t lead = 0;  // opaque: the loads stay behind the branch above
    asm volatile("" : "+v"(lead));
    f32x4v first[16];
    ld16(min((int)threadIdx.x, outs * G - 1), 0, lead, first);
    // a wave per head turns the splits' maxima and sums into weights, 64 splits at a time
    auto ld = [](const float* a) {
        return __hip_atomic_load(a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    __shared__ float wz[NREP][kMaxSplits + 16];
    constexpr int ZR = kMaxSplits / 64;
    for (int r = wave; r < n_rep; r += W) {
        const float* pz = part + ((size_t)t * n_head + kvh * n_rep + r) * S * (HD + 4);
        float m[ZR], l[ZR], M = -INFINITY;
#pragma unroll
        for (int i = 0; i < ZR; ++i) {
            const int zz = 64 * i + lane;
            m[i] = zz < S ? ld(pz + (size_t)zz * (HD + 4) + HD) : -INFINITY;
            l[i] = zz < S ? ld(pz + (size_t)zz * (HD + 4) + HD + 1) : 0.0f;
            M = fmaxf(M, m[i]);
        }
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) M = fmaxf(M, __shfl_xor(M, o, 64));
        float den = 0.0f;
#pragma unroll
        for (int i = 0; i < ZR; ++i) {
            const float e = expf(m[i] - M);
            const float w = m[i] == -INFINITY ? 0.0f : e;
            if (64 * i + lane < S) wz[r][64 * i + lane] = w;
            den = __builtin_fmaf(w, l[i], den);
        }
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) den += __shfl_xor(den, o, 64);
        if (lane == 0) l_all[r] = den;
    }
    __syncthreads();
    for (int o = threadIdx.x; o < outs * G; o += kThreads) {
        const int gi = o / outs, oo = o - gi * outs;
        const int r = oo / Q, d = 4 * (oo - r * Q);
        f32x4v num = {0.0f, 0.0f, 0.0f, 0.0f};
        const int len = min(S, (gi + 1) * zlen) - gi * zlen;
        for (int zz = 0; zz < len; zz += 16) {
            if (zz > 0 || o >= kThreads) ld16(o, zz, 0, first);
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                const float wgt = zz + u < len ? wz[r][gi * zlen + zz + u] : 0.0f;  // past the range: 0 * 0
                num.x = __builtin_fmaf(wgt, first[u].x, num.x);
                num.y = __builtin_fmaf(wgt, first[u].y, num.y);
                num.z = __builtin_fmaf(wgt, first[u].z, num.z);
                num.w = __builtin_fmaf(wgt, first[u].w, num.w);
            }
        }
        if (G == 1) {
            float* op = out + ((size_t)t * n_head + kvh * n_rep + r) * HD + d;
            op[0] = __fdiv_rn(num.x, l_all[r]);
            op[1] = __fdiv_rn(num.y, l_all[r]);
            op[2] = __fdiv_rn(num.z, l_all[r]);
            op[3] = __fdiv_rn(num.w, l_all[r]);
        } else {
            *(f32x4v*)&wpart[gi][4 * oo] = num;
        }
    }
    if (G == 1) return;
    __syncthreads();
    for (int o = threadIdx.x; o < n_rep * HD; o += kThreads) {
        float v = wpart[0][o];
        for (int gi = 1; gi < G; ++gi) v += wpart[gi][o];
        const int r = o / HD, d = o - r * HD;
        out[((size_t)t * n_head + kvh * n_rep + r) * HD + d] = __fdiv_rn(v, l_all[r]);
    }
}

// The split kernel's sequence splits for these rows: enough workgroups for the device, at
// least one chunk per split (one split when the rows' arrival counters would not fit).
int attention_splits(int rows, int pos0, int n_kv) {
    const int L_max = pos0 + rows;
    const int64_t base = (int64_t)n_kv * rows;
    int S = (int)std::min<int64_t>(std::max<int64_t>(1, (512 + base - 1) / base),
                                   (L_max + kChunk - 1) / kChunk);
    S = std::min(S, kMaxSplits);
    if ((int64_t)rows * n_kv > kAttnCounters) S = 1;
    const int split_len = ((L_max + S - 1) / S + kChunk - 1) / kChunk * kChunk;
    return (L_max + split_len - 1) / split_len;
}

template <int HD>
hipError_t launch_attention_hd(const float* q, const float* kc, const float* vc, int rows,
                               int pos0, int n_head, int n_kv, float* out, float* part,
                               size_t part_floats, int* counters, float rope_base, float* k_new,
                               hipStream_t stream) {
    const int L_max = pos0 + rows;
    int S = attention_splits(rows, pos0, n_kv);
    if ((size_t)rows * n_head * S * (HD + 4) > part_floats || !counters) S = 1;
    const int split_len = ((L_max + S - 1) / S + kChunk - 1) / kChunk * kChunk;
    S = (L_max + split_len - 1) / split_len;
    const float scale = 1.0f / std::sqrt((float)HD);  // engine.cpp:121, IEEE on the host
    const int n_rep = n_head / n_kv;
#define CLLM_ATTENTION(R)                                                                        \
    hipLaunchKernelGGL((k_attention<HD, R>), dim3((unsigned)n_kv, (unsigned)rows, (unsigned)S),   \
                       dim3(kThreads), 0, stream, q, kc, vc, n_head, n_kv, pos0, split_len, scale, part, counters,   \
                       out, rope_base, k_new)
    if (n_rep == 1)
        CLLM_ATTENTION(1);
    else if (n_rep == 2)
        CLLM_ATTENTION(2);
    else if (n_rep <= 4)
        CLLM_ATTENTION(4);
    else
        CLLM_ATTENTION(8);
#undef CLLM_ATTENTION
    return hipGetLastError();
}

// ------------------------------------------------------------- many query rows on MFMA

// Prefill attention with fp32's precision: at head_dim 64 and 128 on bf16 MFMA with split operands,
// at head_dim 256 and over caches of 4 GiB and up on the fp32 matrix cores
// (v_mfma_f32_16x16x4f32).
//
// Split operands. K, V, the queries and the probabilities are sums of three bf16 parts (26 bits);
// the six largest of the nine part products leave out at most 2^-24 of a product, as much as an fp32
// product's rounding at most and far less on average, and run 2.7 times as fast as the fp32 MFMA. The scores add the leading products apart from the
// others (8 rounded additions at head_dim 128, where the fp32 form makes 32), and the P.V products
// of 32 positions add up from zero, small ones first, before they join the output. Error against
// 64 bits at 512 rows after 1024 positions (32 + 8 heads of 128): 2.0e-7, the fp32 form's 4.0e-7.
// Queries are split once into LDS; each wave splits its own K and V rows, beside the MFMAs of the
// rows before. What bounds it: that VALU work (about 1200 operations beside 192 MFMAs per 32
// positions and 32 columns) and the loads' way, at two waves per SIMD. MI355X, us, fp32 form against
// this one: 512 rows after 1024 positions 131 / 98, 300 rows 27 / 24.5; 200 rows of 16 + 16 heads
// of 64 13.3 / 12.3. Columns with an output that is not finite are computed again in fp32 (inf * 0
// appears among the parts where fp32 has inf; see attention_pass_f32), and so are those with one
// of less than 2^-90 (see kQueryUp).
//
// Columns. A query block is COLS = 16 * CT (row, head) pairs of one KV head: column c is
// query head c % n_rep of row r0 + c / n_rep, so the n_rep heads of a row and several rows
// share every K and V row loaded.
//
// Balance. Row block b needs pos0 + (its last row + 1) positions, so causal work grows with
// b; a workgroup takes blocks p and n_blocks - 1 - p, and the 16-position steps of the two
// form one list that its W waves split evenly (the wave whose share straddles the two blocks
// works on both). Each wave's part of a block leaves a (max, sum, unnormalised output) partial
// in LDS; one combine at the end adds each block's partials in slot order. The KV head is the
// fastest grid index, which keeps a KV head's workgroups on one XCD (blockIdx modulo 8) and
// its K and V rows in that XCD's L2 when n_kv is 8. Two waves per SIMD (W = 8 up to head_dim
// 128).
//
// One step of the fp32 form, per 16-column tile (the split form: two such score tiles, then P.V
// over their 32 positions): the scores come out transposed, S^T (16 positions x 16
// columns) = K Q^T over HD / 4 MFMAs (lane l holds K row l % 16 and Q column l % 16 at
// dims (HD / 4) (l / 16) + j for MFMA j; even and odd j in two accumulators added at the end,
// which halves the longest rounding chain), so lane l holds column l % 16's scores of
// positions 4 (l / 16) + i in its four result registers. That is the B operand of
// O^T (HD x 16 columns) = V^T P^T, one MFMA per (i, 16-dim tile dt): the A operand is
// V[4 (l / 16) + i][(HD / 16) (l % 16) + dt], dims permuted so each lane reads HD / 16
// consecutive values of a row. The online softmax is per lane: a column's running max and
// sum live in the four lanes l % 16 of its tile, reduced with v_permlane32_swap and
// v_permlane16_swap (lanes l ^ 32, l ^ 16).
//
// Pipeline (fp32 form). A wave issues the next step's score MFMAs interleaved with this step's softmax
// (an MFMA every few VALU instructions, so the matrix pipe stays busy through the softmax),
// then this step's P.V MFMAs; K rows are requested two steps ahead and V rows one step
// ahead. Loads past a part's last step are clamped to rows in bounds instead of branched, so
// a step is one basic block.

// x combined with its value in lanes l ^ 16, l ^ 32 and l ^ 48 (max or sum)
template <bool MAX>
__device__ __forceinline__ float quad_reduce(float x) {
    const unsigned u = __float_as_uint(x);
    const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    const float a0 = __uint_as_float(a[0]), a1 = __uint_as_float(a[1]);
    x = MAX ? fmaxf(a0, a1) : a0 + a1;
    const unsigned v = __float_as_uint(x);
    const auto b = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    const float b0 = __uint_as_float(b[0]), b1 = __uint_as_float(b[1]);
    return MAX ? fmaxf(b0, b1) : b0 + b1;
}

// LDS of a workgroup: the partial outputs, maxima and sums of the parts; while the steps run, the
// split queries lie where the partial outputs of the first waves come later.
template <int HD, int CT, int W>
struct AttnLds {
    static constexpr int COLS = 16 * CT, NS = W + 1, PAD = HD + 4;
    int slot_blk[NS];  // the block (0 or 1) whose partial a slot holds, -1: none
    int bad[2][COLS];  // columns to compute again
    float den[2][COLS], max[2][COLS];
    float m[NS][COLS], l[NS][COLS];
    alignas(16) float o[NS][COLS][PAD];
};

// The matrix cores take bf16 values below 2^-126 for zero, which the lower parts of fp32 values below
// 2^-101 are. The queries are split times this factor: then none is, keys lose less than 2^-53 of a
// score, and queries from 2^66 and scores from 2^66 on overflow and are computed again in fp32.
constexpr float kQueryUp = 0x1p62f;

// One pass over a workgroup's two row blocks; the blocks (bits 0 and 1) where an output of this
// thread is not finite, or so small that lower parts of the values were lost (below 2^-90; values
// that are all below 2^-126 come out as zero).
template <int HD, int CT, int W>
__device__ __forceinline__ int attention_pass(
    AttnLds<HD, CT, W>& sm, const float* __restrict__ q, const float* __restrict__ kc,
    const float* __restrict__ vc, int n_head, int n_kv, int rows, int pos0, int n_blocks, float scale,
    float* __restrict__ out) {
    using Lds = AttnLds<HD, CT, W>;
    constexpr int COLS = Lds::COLS;
    constexpr int DV = HD / 16;  // V values per lane and row
    constexpr int NS = Lds::NS;  // partial slots: one per wave, one more for the straddling wave
    constexpr int SP = 32;       // positions per step
    auto& o_sm = sm.o;
    auto& m_sm = sm.m;
    auto& l_sm = sm.l;
    auto& den_sm = sm.den;
    auto& slot_blk = sm.slot_blk;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col16 = lane & 15, quad = lane >> 4;
    const int g = blockIdx.x % n_kv, pair = blockIdx.x / n_kv;
    const int n_rep = n_head / n_kv, rpb = COLS / n_rep, used = rpb * n_rep;
    const size_t kv_dim = (size_t)n_kv * HD;

    const int blk_row[2] = {pair * rpb, (n_blocks - 1 - pair) * rpb};
    const bool two = n_blocks - 1 - pair > pair;
    const int len[2] = {pos0 + min(rows, blk_row[0] + rpb), two ? pos0 + min(rows, blk_row[1] + rpb) : 0};
    const int nA = (len[0] + SP - 1) / SP, T = nA + (len[1] + SP - 1) / SP;
    const int g0 = wave * T / W, g1 = (wave + 1) * T / W;
    if (lane == 0) {
        slot_blk[wave] = g0 >= g1 ? -1 : g1 > nA ? 1 : 0;
        if (wave == 0) {
            bool straddle = false;
            for (int w = 0; w < W; ++w) straddle |= w * T / W < nA && nA < (w + 1) * T / W;
            slot_blk[W] = straddle ? 0 : -1;
        }
    }

    // the columns of both blocks as three bf16 parts, [block][part][column][HD], 16-byte
    // chunk c of a column at slot c ^ (column & 7)
    if (threadIdx.x < 2 * COLS) sm.bad[threadIdx.x / COLS][threadIdx.x % COLS] = 0;
    uint8_t* qlds = (uint8_t*)sm.o;
    constexpr int QCOL = HD * 2, QPART = COLS * QCOL;
    static_assert(6 * QPART <= W * COLS * Lds::PAD * 4, "the queries end below the straddling wave's slot");
    {
        for (int i = threadIdx.x; i < 2 * COLS * (HD / 8); i += W * 64) {
            const int blk = i / (COLS * (HD / 8)), c = (i / (HD / 8)) % COLS, ch = i % (HD / 8);
            const int t = blk_row[blk] + c / n_rep;
            const bool valid = c < used && t < rows;  // unused columns: zeros
            const float* qr = q + ((size_t)min(t, rows - 1) * n_head + g * n_rep + c % n_rep) * HD + 8 * ch;
            const f32x4 v0 = *(const f32x4*)qr, v1 = *(const f32x4*)(qr + 4);
            float v[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = valid ? v[e] * kQueryUp : 0.0f;
            wbf8 p[3];
            split8<3>(v, p);
#pragma unroll
            for (int u = 0; u < 3; ++u)
                *(wbf8*)(qlds + (blk * 3 + u) * QPART + c * QCOL + ((ch ^ (c & 7)) << 4)) = p[u];
        }
        __syncthreads();
    }

    // a part's partial: result register r of dim tile dt is dim DV (4 (l / 16) + r) + dt of
    // column l % 16, so each lane stores HD / 4 consecutive dims
    auto store_partial = [&](int slot, const f32x4 (&o)[CT][DV], const float (&m_run)[CT], const float (&l_run)[CT]) {
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            const int c = ct * 16 + col16;
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int dt = 0; dt < DV; ++dt) o_sm[slot][c][DV * (4 * quad + r) + dt] = o[ct][dt][r];
            if (quad == 0) {
                m_sm[slot][c] = m_run[ct];
                l_sm[slot][c] = l_run[ct];
            }
        }
    };

    // one wave's share of a block; false where it has none
    auto run_part = [&](int part, f32x4 (&o)[CT][DV], float (&m_run)[CT], float (&l_run)[CT]) {
        const int s0 = part == 0 ? g0 : max(g0, nA) - nA;
        const int s1 = part == 0 ? min(g1, nA) : g1 - nA;
        if (s0 >= s1) return false;
        const int r0 = blk_row[part], L = len[part];

        // the last position a column sees (-1: an unused column, every score masked)
        int lim[CT];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            const int c = ct * 16 + col16, t = r0 + c / n_rep;
            lim[ct] = c < used && t < rows ? pos0 + t : -1;
        }
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            m_run[ct] = -INFINITY;
            l_run[ct] = 0.0f;
#pragma unroll
            for (int dt = 0; dt < DV; ++dt) o[ct][dt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }

        // K rows 32 s + 16 u + l % 16 (dims 32 ks + 8 (l / 16) + e), V rows 32 s + 4 (l / 16) +
        // i and 16 more (dims DV (l % 16) + d), positions and steps clamped as below
        constexpr int KS = HD / 32, VH = DV / 4;
        float kf[2][8 * KS], vf[VH][8][4];
        // byte offsets of 32 bits (the host takes the fp32 pass for caches of 4 GiB and up)
        const uint32_t row4 = 4u * (uint32_t)kv_dim;
        const uint32_t k_at = 4u * (uint32_t)(g * HD + 8 * quad), v_at = 4u * (uint32_t)(g * HD + DV * col16);
        auto load_k = [&](int s, int u) {
            const uint32_t at = (uint32_t)min(min(s, s1 - 1) * 32 + 16 * u + col16, L - 1) * row4 + k_at;
#pragma unroll
            for (int j = 0; j < 2 * KS; ++j) {
                const f32x4 v = *(const f32x4*)((const char*)kc + at + (128 * (j >> 1) + 16 * (j & 1)));
                kf[u][4 * j] = v.x; kf[u][4 * j + 1] = v.y; kf[u][4 * j + 2] = v.z; kf[u][4 * j + 3] = v.w;
            }
        };
        auto load_v = [&](int s, int hf) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int p = min(s, s1 - 1) * 32 + (e < 4 ? 0 : 16) + 4 * quad + (e & 3);
                const f32x4 v = *(const f32x4*)((const char*)vc + ((uint32_t)min(p, L - 1) * row4 + v_at) + 16 * hf);
                vf[hf][e][0] = v.x; vf[hf][e][1] = v.y; vf[hf][e][2] = v.z; vf[hf][e][3] = v.w;
            }
        };
        const uint8_t* qb = qlds + part * 3 * QPART + col16 * QCOL;
        load_k(s0, 0);
        for (int s = s0; s < s1; ++s) {
            // the scores, transposed: 16 positions x 16 columns per (u, ct). Loads go out one
            // phase (half of the scores, half of P.V) ahead of their use.
            f32x4 sc[2][CT];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                __builtin_amdgcn_sched_barrier(0);
                if (u == 0)
                    load_k(s, 1);
                else
                    load_v(s, 0);
                f32x4 hi[CT], lo[CT];
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) hi[ct] = lo[ct] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                // the next K step is split beside this one's MFMAs
                wbf8 kps[2][3];
                split8<3>(&kf[u][0], kps[0]);
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    __builtin_amdgcn_sched_barrier(0);
                    if (ks + 1 < KS) split8<3>(&kf[u][8 * (ks + 1)], kps[(ks + 1) & 1]);
                    const wbf8 (&kp)[3] = kps[ks & 1];
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct) {
                        const uint8_t* p = qb + ct * 16 * QCOL + (((4 * ks + quad) ^ (col16 & 7)) << 4);
                        const wbf8 q0 = *(const wbf8*)p, q1 = *(const wbf8*)(p + QPART);
                        const wbf8 q2 = *(const wbf8*)(p + 2 * QPART);
                        lo[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kp[2], q0, lo[ct], 0, 0, 0);
                        hi[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kp[0], q0, hi[ct], 0, 0, 0);
                        lo[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kp[0], q2, lo[ct], 0, 0, 0);
                        lo[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kp[1], q1, lo[ct], 0, 0, 0);
                        lo[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kp[1], q0, lo[ct], 0, 0, 0);
                        lo[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kp[0], q1, lo[ct], 0, 0, 0);
                    }
                    __builtin_amdgcn_sched_group_barrier(0x100, 3 * CT, 0);
#pragma unroll
                    for (int i = 0; i < 6 * CT; ++i) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // an MFMA
                        __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);  // VALU beside it
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) sc[u][ct] = hi[ct] + lo[ct];
            }
            __builtin_amdgcn_sched_barrier(0);
            // the online softmax of the step's 32 positions, as below
            wbf8 pp[CT][3];
            float cr[CT];
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                float sv[8], pr[8], mx = -INFINITY;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int p = s * 32 + (e < 4 ? 0 : 16) + 4 * quad + (e & 3);
                    sv[e] = p <= lim[ct] ? __fmul_rn(sc[e >> 2][ct][e & 3], scale / kQueryUp) : -INFINITY;
                    mx = fmaxf(mx, sv[e]);
                }
                mx = quad_reduce<true>(mx);
                const float mo = m_run[ct], mn = fmaxf(mo, mx);
                float ps = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float x = expf(sv[e] - mn);
                    pr[e] = sv[e] == -INFINITY ? 0.0f : x;
                    ps += pr[e];
                }
                ps = quad_reduce<false>(ps);
                const float x = expf(mo - mn);
                cr[ct] = mo == -INFINITY ? 0.0f : x;
                m_run[ct] = mn;
                l_run[ct] = __builtin_fmaf(l_run[ct], cr[ct], ps);
                split8<3>(pr, pp[ct]);
            }
            // P.V of 32 positions per dim tile, small products first, then into the output
#pragma unroll
            for (int hf = 0; hf < VH; ++hf) {
                __builtin_amdgcn_sched_barrier(0);
                if (hf + 1 < VH)
                    load_v(s, hf + 1);
                else
                    load_k(s + 1, 0);
                wbf8 vps[2][3];
                auto split_v = [&](int d, wbf8 (&p)[3]) {
                    float v[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[e] = vf[hf][e][d];
                    split8<3>(v, p);
                };
                split_v(0, vps[0]);
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    __builtin_amdgcn_sched_barrier(0);
                    if (d + 1 < 4) split_v(d + 1, vps[(d + 1) & 1]);
                    const wbf8 (&vp)[3] = vps[d & 1];
                    f32x4 t[CT];
                    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct) t[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vp[2], pp[ct][0], zero, 0, 0, 0);
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct) t[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vp[0], pp[ct][2], t[ct], 0, 0, 0);
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct) t[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vp[1], pp[ct][1], t[ct], 0, 0, 0);
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct) t[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vp[1], pp[ct][0], t[ct], 0, 0, 0);
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct) t[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vp[0], pp[ct][1], t[ct], 0, 0, 0);
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct) t[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vp[0], pp[ct][0], t[ct], 0, 0, 0);
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            o[ct][4 * hf + d][r] = __builtin_fmaf(o[ct][4 * hf + d][r], cr[ct], t[ct][r]);
#pragma unroll
                    for (int i = 0; i < 6 * CT; ++i) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
                    }
                }
            }
        }
        return true;
    };
    // the straddling wave's first part goes to its slot at once; the others wait until the queries
    // are read no more
    f32x4 o[CT][DV];
    float m_run[CT], l_run[CT];
    for (int part = 0; part < 2; ++part)
        if (run_part(part, o, m_run, l_run) && part == 0 && g1 > nA) store_partial(W, o, m_run, l_run);
    __syncthreads();
    if (g0 < g1) store_partial(wave, o, m_run, l_run);
    __syncthreads();
    // per (block, column): the partials' weights e^(m - M) in place of their maxima, and the sum
    if (threadIdx.x < 2 * COLS) {
        const int blk = threadIdx.x / COLS, c = threadIdx.x % COLS;
        float M = -INFINITY;
        for (int z = 0; z < NS; ++z)
            if (slot_blk[z] == blk) M = fmaxf(M, m_sm[z][c]);
        float den = 0.0f;
        for (int z = 0; z < NS; ++z) {
            if (slot_blk[z] != blk) continue;
            const float m = m_sm[z][c];
            const float e = expf(m - M);
            const float wgt = m == -INFINITY ? 0.0f : e;
            den = __builtin_fmaf(wgt, l_sm[z][c], den);
            m_sm[z][c] = wgt;
        }
        den_sm[blk][c] = den;
    }
    __syncthreads();
    int bad = 0;
    for (int o4 = threadIdx.x; o4 < 2 * COLS * (HD / 4); o4 += W * 64) {
        const int blk = o4 / (COLS * (HD / 4));
        const int c = (o4 / (HD / 4)) % COLS, d = (o4 % (HD / 4)) * 4;
        const int t = blk_row[blk] + c / n_rep;
        if ((blk == 1 && !two) || c >= used || t >= rows) continue;
        f32x4 num = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        for (int z = 0; z < NS; ++z) {
            if (slot_blk[z] != blk) continue;
            const float wgt = m_sm[z][c];
            const f32x4 v = *(const f32x4*)&o_sm[z][c][d];
            num.x = __builtin_fmaf(wgt, v.x, num.x);
            num.y = __builtin_fmaf(wgt, v.y, num.y);
            num.z = __builtin_fmaf(wgt, v.z, num.z);
            num.w = __builtin_fmaf(wgt, v.w, num.w);
        }
        const float den = den_sm[blk][c];
        const f32x4 res = f32x4{__fdiv_rn(num.x, den), __fdiv_rn(num.y, den), __fdiv_rn(num.z, den), __fdiv_rn(num.w, den)};
        // (a magnitude between them, or zero; NaN is neither)
        const auto sound = [](float v) { return (fabsf(v) < INFINITY && fabsf(v) >= 0x1p-90f) || v == 0.0f; };
        if (!(sound(res.x) && sound(res.y) && sound(res.z) && sound(res.w))) {
            sm.bad[blk][c] = 1;
            bad |= 1 << blk;
        }
        float* orow = out + ((size_t)t * n_head + g * n_rep + c % n_rep) * HD + d;
        orow[0] = res.x;  // out is 4-byte aligned only
        orow[1] = res.y;
        orow[2] = res.z;
        orow[3] = res.w;
    }
    return bad;
}

// Positions [p0, p1) of one column, a wave's lanes over the dims (lane + 64 e), four positions at a
// time, on top of its output o, maximum m and sum l so far.
template <int HD>
__device__ __forceinline__ void attention_tail(const float* qr, const float* kr, const float* vr,
                                               size_t kv_dim, int p0, int p1, float scale,
                                               float (&o)[HD / 64], float& m, float& l) {
    constexpr int E = HD / 64;
    const int lane = threadIdx.x & 63;
    float qv[E];
#pragma unroll
    for (int e = 0; e < E; ++e) qv[e] = qr[lane + 64 * e];
    for (int p = p0; p < p1; p += 4) {
        float s[4], v[4][E], mx = m;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const size_t at = (size_t)min(p + i, p1 - 1) * kv_dim + lane;
            s[i] = 0.0f;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                s[i] = __builtin_fmaf(qv[e], kr[at + 64 * e], s[i]);
                v[i][e] = vr[at + 64 * e];
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int j = 32; j >= 1; j >>= 1) s[i] += __shfl_xor(s[i], j, 64);
            s[i] = p + i < p1 ? __fmul_rn(s[i], scale) : -INFINITY;
            mx = fmaxf(mx, s[i]);
        }
        const float x = expf(m - mx), cr = m == -INFINITY ? 0.0f : x;
        l *= cr;
#pragma unroll
        for (int e = 0; e < E; ++e) o[e] *= cr;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float y = expf(s[i] - mx), pr = s[i] == -INFINITY ? 0.0f : y;
            l += pr;
#pragma unroll
            for (int e = 0; e < E; ++e) o[e] = p + i < p1 ? __builtin_fmaf(pr, v[i][e], o[e]) : o[e];
        }
        m = mx;
    }
}

// The fp32 form of a pass. REDO: only the columns of sm.bad, of the blocks of redo (bits 0 and 1).
// Their MFMA steps then stop at the last whole one that every column of the block sees, and each
// column's remaining positions (at most 16 and the block's rows) go by themselves: a position that
// a column does not see is not multiplied by a probability of zero, which an infinite value would
// make NaN.
template <int HD, int CT, int W, bool REDO>
__device__ __forceinline__ void attention_pass_f32(
    AttnLds<HD, CT, W>& sm, const float* __restrict__ q, const float* __restrict__ kc,
    const float* __restrict__ vc, int n_head, int n_kv, int rows, int pos0, int n_blocks, float scale,
    float* __restrict__ out, int redo) {
    using Lds = AttnLds<HD, CT, W>;
    constexpr int COLS = Lds::COLS;
    constexpr int DQ = HD / 4;   // K and Q values per lane and row
    constexpr int DV = HD / 16;  // V values per lane and row
    constexpr int NS = Lds::NS;  // partial slots: one per wave, one more for the straddling wave
    auto& o_sm = sm.o;
    auto& m_sm = sm.m;
    auto& l_sm = sm.l;
    auto& den_sm = sm.den;
    auto& slot_blk = sm.slot_blk;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col16 = lane & 15, quad = lane >> 4;
    const int g = blockIdx.x % n_kv, pair = blockIdx.x / n_kv;
    const int n_rep = n_head / n_kv, rpb = COLS / n_rep, used = rpb * n_rep;
    const size_t kv_dim = (size_t)n_kv * HD;
    const float* kg = kc + (size_t)g * HD + DQ * quad;
    const float* vg = vc + (size_t)g * HD + DV * col16;

    const int blk_row[2] = {pair * rpb, (n_blocks - 1 - pair) * rpb};
    const bool two = n_blocks - 1 - pair > pair;
    const int len[2] = {
        !REDO ? pos0 + min(rows, blk_row[0] + rpb) : redo & 1 ? (pos0 + blk_row[0] + 1) & ~15 : 0,
        !two ? 0 : !REDO ? pos0 + min(rows, blk_row[1] + rpb) : redo & 2 ? (pos0 + blk_row[1] + 1) & ~15 : 0};
    const int nA = (len[0] + 15) / 16, T = nA + (len[1] + 15) / 16;
    const int g0 = wave * T / W, g1 = (wave + 1) * T / W;
    if (lane == 0) {
        slot_blk[wave] = g0 >= g1 ? -1 : g1 > nA ? 1 : 0;
        if (wave == 0) {
            bool straddle = false;
            for (int w = 0; w < W; ++w) straddle |= w * T / W < nA && nA < (w + 1) * T / W;
            slot_blk[W] = straddle ? 0 : -1;
        }
    }

    for (int part = 0; part < 2; ++part) {
        const int s0 = part == 0 ? g0 : max(g0, nA) - nA;
        const int s1 = part == 0 ? min(g1, nA) : g1 - nA;
        if (s0 >= s1) continue;
        const int r0 = blk_row[part], L = len[part];
        const int slot = part == 0 && g1 > nA ? W : wave;

        // the queries of this lane's columns (unused columns: zeros from a row in bounds);
        // lim = the last position a column sees (-1: an unused column, every score masked)
        float qf[CT][DQ];
        int lim[CT];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            const int c = ct * 16 + col16;
            const int t = r0 + c / n_rep;
            const bool valid = c < used && t < rows;
            lim[ct] = valid ? pos0 + t : -1;
            const float* qr = q + ((size_t)min(t, rows - 1) * n_head + g * n_rep + c % n_rep) * HD + DQ * quad;
#pragma unroll
            for (int j = 0; j < DQ; j += 4) {
                const f32x4 v = *(const f32x4*)(qr + j);
                qf[ct][j] = valid ? v.x : 0.0f;
                qf[ct][j + 1] = valid ? v.y : 0.0f;
                qf[ct][j + 2] = valid ? v.z : 0.0f;
                qf[ct][j + 3] = valid ? v.w : 0.0f;
            }
        }
        f32x4 o[CT][DV];
        float m_run[CT], l_run[CT];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            m_run[ct] = -INFINITY;
            l_run[ct] = 0.0f;
#pragma unroll
            for (int dt = 0; dt < DV; ++dt) o[ct][dt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }

        // K row 16 s + l % 16 and V rows 16 s + 4 (l / 16) + i of step s, positions clamped
        // to the block's last (their scores are masked) and steps to the part's last
        float kf[DQ], vf[4][DV];
        auto load_k = [&](int s) {
            const float* kr = kg + (size_t)min(min(s, s1 - 1) * 16 + col16, L - 1) * kv_dim;
#pragma unroll
            for (int j = 0; j < DQ; j += 4) {
                const f32x4 v = *(const f32x4*)(kr + j);
                kf[j] = v.x; kf[j + 1] = v.y; kf[j + 2] = v.z; kf[j + 3] = v.w;
            }
        };
        auto load_v = [&](int s) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float* vr = vg + (size_t)min(min(s, s1 - 1) * 16 + 4 * quad + i, L - 1) * kv_dim;
#pragma unroll
                for (int e = 0; e < DV; e += 4) {
                    const f32x4 v = *(const f32x4*)(vr + e);
                    vf[i][e] = v.x; vf[i][e + 1] = v.y; vf[i][e + 2] = v.z; vf[i][e + 3] = v.w;
                }
            }
        };
        auto scores = [&](f32x4 (&sa)[CT][2]) {
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) sa[ct][0] = sa[ct][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int j = 0; j < DQ; ++j)
#pragma unroll
                for (int ct = 0; ct < CT; ++ct)
                    sa[ct][j & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[j], qf[ct][j], sa[ct][j & 1], 0, 0, 0);
        };
        // the online softmax of step s's scores: probabilities into pr, the running max, sum
        // and output rescaled (by exactly 1 while a column's max stands)
        float pr[CT][4];
        auto softmax = [&](int s, const f32x4 (&sa)[CT][2]) {
            const int pq = s * 16 + 4 * quad;  // position of result register 0
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                const f32x4 sc = sa[ct][0] + sa[ct][1];
                float sv[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) sv[i] = pq + i <= lim[ct] ? __fmul_rn(sc[i], scale) : -INFINITY;
                const float mx = quad_reduce<true>(fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3])));
                const float mo = m_run[ct], mn = fmaxf(mo, mx);
                float ps = 0.0f;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float e = expf(sv[i] - mn);
                    pr[ct][i] = sv[i] == -INFINITY ? 0.0f : e;
                    ps += pr[ct][i];
                }
                ps = quad_reduce<false>(ps);
                const float e = expf(mo - mn);
                const float cr = mo == -INFINITY ? 0.0f : e;
                m_run[ct] = mn;
                l_run[ct] = __builtin_fmaf(l_run[ct], cr, ps);
#pragma unroll
                for (int dt = 0; dt < DV; ++dt) o[ct][dt] *= cr;
            }
        };
        auto pv = [&]() {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int dt = 0; dt < DV; ++dt)
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct)
                        o[ct][dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[i][dt], pr[ct][i], o[ct][dt], 0, 0, 0);
        };

        f32x4 sa[CT][2];
        load_k(s0);
        load_v(s0);
        if constexpr (REDO) {  // (one step at a time: no registers for a second beside the first pass's)
#pragma unroll 1
            for (int s = s0; s < s1 - 1; ++s) {
                scores(sa);
                load_k(s + 1);
                softmax(s, sa);
                pv();
                load_v(s + 1);
            }
            scores(sa);
        } else {
            scores(sa);
            load_k(s0 + 1);
            for (int s = s0; s < s1 - 1; ++s) {
                f32x4 sn[CT][2];
                scores(sn);        // step s + 1 (K rows requested a step ago)
                load_k(s + 2);
                softmax(s, sa);    // step s, beside the score MFMAs
#pragma unroll
                for (int i = 0; i < DQ * CT; ++i) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
                    __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);  // five VALU
                }
                pv();
                // (not among the MFMAs that read the old rows: the copies that takes cost 8 % at
                // head_dim 256, 320 rows of 8 + 8 heads after 1024 positions 120 against 111 us)
                __builtin_amdgcn_sched_barrier(0);
                load_v(s + 1);     // V rows a step ahead of their P.V MFMAs
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) {
                    sa[ct][0] = sn[ct][0];
                    sa[ct][1] = sn[ct][1];
                }
            }
        }
        softmax(s1 - 1, sa);
        pv();

        // the part's partial: result register r of dim tile dt is dim DV (4 (l / 16) + r) + dt
        // of column l % 16, so each lane stores HD / 4 consecutive dims
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            const int c = ct * 16 + col16;
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int dt = 0; dt < DV; ++dt) o_sm[slot][c][DV * (4 * quad + r) + dt] = o[ct][dt][r];
            if (quad == 0) {
                m_sm[slot][c] = m_run[ct];
                l_sm[slot][c] = l_run[ct];
            }
        }
    }
    __syncthreads();
    // per (block, column): the partials' weights e^(m - M) in place of their maxima, and the sum
    if (threadIdx.x < 2 * COLS) {
        const int blk = threadIdx.x / COLS, c = threadIdx.x % COLS;
        float M = -INFINITY;
        for (int z = 0; z < NS; ++z)
            if (slot_blk[z] == blk) M = fmaxf(M, m_sm[z][c]);
        float den = 0.0f;
        for (int z = 0; z < NS; ++z) {
            if (slot_blk[z] != blk) continue;
            const float m = m_sm[z][c];
            const float e = expf(m - M);
            const float wgt = m == -INFINITY ? 0.0f : e;
            den = __builtin_fmaf(wgt, l_sm[z][c], den);
            m_sm[z][c] = wgt;
        }
        den_sm[blk][c] = den;
        if constexpr (REDO) sm.max[blk][c] = M;
    }
    __syncthreads();
    if constexpr (REDO) {
        constexpr int E = HD / 64;
        for (int i = wave; i < 2 * COLS; i += W) {
            const int blk = i / COLS, c = i % COLS, t = blk_row[blk] + c / n_rep;
            if (!__builtin_amdgcn_readfirstlane(sm.bad[blk][c])) continue;
            float o[E], m = sm.max[blk][c], l = den_sm[blk][c];
#pragma unroll
            for (int e = 0; e < E; ++e) o[e] = 0.0f;
            for (int z = 0; z < NS; ++z) {
                if (slot_blk[z] != blk) continue;
                const float wgt = m_sm[z][c];
#pragma unroll
                for (int e = 0; e < E; ++e) o[e] = __builtin_fmaf(wgt, o_sm[z][c][lane + 64 * e], o[e]);
            }
            const size_t at = ((size_t)t * n_head + g * n_rep + c % n_rep) * HD;
            attention_tail<HD>(q + at, kc + (size_t)g * HD, vc + (size_t)g * HD, kv_dim, len[blk], pos0 + t + 1, scale,
                               o, m, l);
#pragma unroll
            for (int e = 0; e < E; ++e) out[at + lane + 64 * e] = __fdiv_rn(o[e], l);
        }
        return;
    }
    for (int o4 = threadIdx.x; o4 < 2 * COLS * (HD / 4); o4 += W * 64) {
        const int blk = o4 / (COLS * (HD / 4));
        const int c = (o4 / (HD / 4)) % COLS, d = (o4 % (HD / 4)) * 4;
        const int t = blk_row[blk] + c / n_rep;
        if ((blk == 1 && !two) || c >= used || t >= rows) continue;
        f32x4 num = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        for (int z = 0; z < NS; ++z) {
            if (slot_blk[z] != blk) continue;
            const float wgt = m_sm[z][c];
            const f32x4 v = *(const f32x4*)&o_sm[z][c][d];
            num.x = __builtin_fmaf(wgt, v.x, num.x);
            num.y = __builtin_fmaf(wgt, v.y, num.y);
            num.z = __builtin_fmaf(wgt, v.z, num.z);
            num.w = __builtin_fmaf(wgt, v.w, num.w);
        }
        const float den = den_sm[blk][c];
        float* orow = out + ((size_t)t * n_head + g * n_rep + c % n_rep) * HD + d;
        orow[0] = __fdiv_rn(num.x, den);  // out is 4-byte aligned only
        orow[1] = __fdiv_rn(num.y, den);
        orow[2] = __fdiv_rn(num.z, den);
        orow[3] = __fdiv_rn(num.w, den);
    }
}

// The fp32 form at head_dim 256, the split operands at 64 and 128. A column with an output that is
// not finite is computed again in fp32 (inf * 0 appears among the parts where fp32 has inf); the
// others keep their bits. A batch that is NaN throughout takes the time of both forms and of the
// tails: 512 rows of 32 + 8 heads of 128 after 1024 positions 235 us, 98 when finite (one
// position at a time and column after column, all columns of the workgroup: 4000).
template <int HD, int CT, int W>
__global__ __launch_bounds__(W * 64) void k_attention_mfma(
    const float* __restrict__ q, const float* __restrict__ kc, const float* __restrict__ vc,
    int n_head, int n_kv, int rows, int pos0, int n_blocks, float scale, float* __restrict__ out) {
    if constexpr (HD == 256) {
        __shared__ AttnLds<HD, CT, W> sm;
        attention_pass_f32<HD, CT, W, false>(sm, q, kc, vc, n_head, n_kv, rows, pos0, n_blocks, scale, out, 0);
    } else {
        extern __shared__ __align__(16) uint8_t attn_lds[];
        auto& sm = *(AttnLds<HD, CT, W>*)attn_lds;
        const int bad = attention_pass<HD, CT, W>(sm, q, kc, vc, n_head, n_kv, rows, pos0, n_blocks, scale, out);
        if (!__syncthreads_or(bad)) return;
        const int redo = (__syncthreads_or(bad & 1) ? 1 : 0) | (__syncthreads_or(bad & 2) ? 2 : 0);
        attention_pass_f32<HD, CT, W, true>(sm, q, kc, vc, n_head, n_kv, rows, pos0, n_blocks, scale, out, redo);
    }
}

// Caches past the split operands' 32-bit offsets.
template <int HD, int CT, int W>
__global__ __launch_bounds__(W * 64) void k_attention_mfma_f32(
    const float* __restrict__ q, const float* __restrict__ kc, const float* __restrict__ vc,
    int n_head, int n_kv, int rows, int pos0, int n_blocks, float scale, float* __restrict__ out) {
    __shared__ AttnLds<HD, CT, W> sm;
    attention_pass_f32<HD, CT, W, false>(sm, q, kc, vc, n_head, n_kv, rows, pos0, n_blocks, scale, out, 0);
}

// Whether the caches are past the split operands' 32-bit offsets.
bool attention_large_cache(int rows, int pos0, int n_kv, int head_dim) {
    return ((uint64_t)pos0 + (uint64_t)rows) * (uint64_t)n_kv * (uint64_t)head_dim * sizeof(float) >= (1ull << 32);
}

template <int HD, int CT, int W>
hipError_t launch_attention_mfma_hd(const float* q, const float* kc, const float* vc, int rows,
                                    int pos0, int n_head, int n_kv, float* out, hipStream_t stream) {
    const int rpb = 16 * CT / (n_head / n_kv);
    const int n_blocks = (rows + rpb - 1) / rpb;
    const int pairs = (n_blocks + 1) / 2;
    const float scale = 1.0f / std::sqrt((float)HD);  // engine.cpp:121, IEEE on the host
    const dim3 grid((unsigned)(n_kv * pairs));
    int lds = 0;  // of head_dim 256, static
    if constexpr (HD <= 128) {
        if (attention_large_cache(rows, pos0, n_kv, HD)) {
            hipLaunchKernelGGL((k_attention_mfma_f32<HD, CT, W>), grid, dim3(W * 64), 0, stream, q, kc, vc, n_head,
                               n_kv, rows, pos0, n_blocks, scale, out);
            return hipGetLastError();
        }
        lds = sizeof(AttnLds<HD, CT, W>);
        static_assert(sizeof(AttnLds<HD, CT, W>) <= 160 * 1024, "LDS budget");
        static LdsLimit limit;
        const hipError_t e = limit.raise((const void*)k_attention_mfma<HD, CT, W>, lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((k_attention_mfma<HD, CT, W>), grid, dim3(W * 64), lds, stream, q, kc, vc, n_head, n_kv,
                       rows, pos0, n_blocks, scale, out);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_rope_neox(float* x, int rows, int n_heads, float* x2, int n_heads2,
                            int head_dim, int pos0, float base, hipStream_t stream) {
    if (!x2) n_heads2 = 0;
    if (rows <= 0 || n_heads + n_heads2 <= 0) return hipSuccess;
    if (head_dim <= 0 || head_dim % 2 != 0 || head_dim > 512) return hipErrorInvalidValue;
    const int groups = (n_heads + n_heads2 + kRopeHeads - 1) / kRopeHeads;
    hipLaunchKernelGGL(k_rope_neox, dim3((unsigned)rows, (unsigned)groups), dim3(256),
                       0, stream, x, n_heads, x2, n_heads2, head_dim, pos0, base);
    return hipGetLastError();
}

size_t attention_workspace_bytes(int rows, int n_head, int head_dim) {
    // attention_splits: at most 512 / (n_kv * rows) + 1 splits, n_kv >= 1
    const size_t splits = (size_t)(512 / std::max(rows, 1) + 1);
    return kAttnCounters * sizeof(int) + (size_t)rows * n_head * splits * (head_dim + 4) * sizeof(float);
}

namespace {

// Row blocks of the MFMA kernel (16 CT columns, rpb whole rows each) and its workgroups: n_kv x
// pairs of blocks.
struct MfmaGrid {
    int rpb, blocks, groups;
};
MfmaGrid attention_mfma_grid(int rows, int n_head, int n_kv, int head_dim) {
    const int rpb = 16 * (head_dim == 256 ? 1 : 2) / (n_head / n_kv);
    const int blocks = (rows + rpb - 1) / rpb;
    return {rpb, blocks, n_kv * ((blocks + 1) / 2)};
}

}  // namespace

// Which kernel: the split kernel's work grows with the rows (each reads its KV head's cache rows
// anew, from L2), the MFMA kernel's time hardly does while its workgroups fit the CUs.
//
// From three query heads per KV head: the MFMA kernel (no workspace, no sequence split) from 33
// rows where it has 32 workgroups (49 rows at 8 KV heads of 4 query heads). MI355X, head_dim 128,
// us, split against MFMA kernel: 32 rows of 32 + 8 heads at the end of 1024 positions 24 / 69, of
// 4096 67 / 220; 64 rows of 64 + 16 heads at 4096 229 / 223, of 128 + 32 heads at 1024 114 / 70.
// Over up to 112 positions (head_dim 64 and 128) the MFMA kernel's waves have one step or none and
// wait for its loads one after the other, so fewer rows stay on the split kernel: 96 rows of 32 + 8 heads 12.3 / 16.1,
// 48 of 64 + 8 10.3 / 14.7, of 64 + 16 11.6 / 14.9 (80 rows 17.6 / 16.1); not 64 rows over 64
// positions, two whole steps, which take 12.6 on either.
//
// One or two query heads per KV head, up to 128 rows (256 at head_dim 256; more take the MFMA
// kernel): the faster by two measured rates. The split kernel reads rows x n_kv x positions K and
// V rows at 32 TB/s, with about as much as 64 positions take for the ends of each workgroup; the
// waves of an MFMA workgroup share the steps over its two blocks' positions and take 4.2 / 6.5 /
// 3.0 us for one (32 positions at head_dim 64 and 128, 16 at 256). MI355X, us, split against MFMA kernel at 64 + 64 heads of 128: 32 rows after 4096
// positions 364 / 117, 8 rows 90 / 117, 128 rows after 1024 368 / 71, 24 rows over 24 9 / 11; 16 + 16
// heads of 64, 128 rows after 256 17 / 21, after 4096 160 / 138; 128 rows of 8 + 4 heads of 256
// after 1024 55 / 103, of 32 + 32 319 / 115.
bool attention_uses_mfma(int rows, int pos0, int n_head, int n_kv, int head_dim) {
    const int kind = tuning().attention_kind.load();
    if (kind != 0) return kind == 2;
    const int n_rep = n_head / n_kv;
    const MfmaGrid g = attention_mfma_grid(rows, n_head, n_kv, head_dim);
    const int positions = pos0 + rows;
    if (n_rep > 2) {
        const int few = head_dim == 256 ? 0 : n_rep <= 4 ? 960 : positions < 64 ? 512 : 0;
        if (positions <= 112 && positions != 64 && rows * n_kv < few) return false;
        return rows > 32 && g.groups >= 32;
    }
    if (rows > (head_dim == 256 ? 256 : 128)) return g.groups >= 32;
    const float split_us = (float)rows * n_kv * (pos0 + 0.5f * rows + 64.0f) * (8.0f * head_dim) / 32e6f;
    const int step = head_dim == 256 ? 16 : 32, waves = head_dim == 256 ? 4 : 8;
    const float start_us = head_dim == 64 ? 0.0f : 2.0f;  // beyond the split kernel's
    const float step_us = head_dim == 64 ? 4.2f : head_dim == 128 ? 6.5f : 3.0f;
    const int steps = (pos0 + std::min(rows, g.rpb) + step - 1) / step +
                      (g.blocks > 1 ? (positions + step - 1) / step : 0);
    const int rounds = (g.groups + 255) / 256;
    return split_us > start_us + step_us * (float)((steps + waves - 1) / waves * rounds);
}

void attention_plan_name(int rows, int pos0, int n_head, int n_kv, int head_dim, char* buf,
                         size_t cap) {
    if (attention_uses_mfma(rows, pos0, n_head, n_kv, head_dim)) {
        const int ct = head_dim == 256 ? 1 : 2, w = head_dim == 256 ? 4 : 8;
        const bool f32 = head_dim != 256 && attention_large_cache(rows, pos0, n_kv, head_dim);
        snprintf(buf, cap, "k_attention_mfma%s<%d,%d,%d> workgroups=%d", f32 ? "_f32" : "", head_dim, ct, w,
                 attention_mfma_grid(rows, n_head, n_kv, head_dim).groups);
    } else {
        snprintf(buf, cap, "k_attention<%d> splits=%d", head_dim, attention_splits(rows, pos0, n_kv));
    }
}

bool attention_supported(int head_dim, int n_head, int n_kv) {
    return (head_dim == 64 || head_dim == 128 || head_dim == 256) && n_kv > 0 &&
           n_head % n_kv == 0 && n_head / n_kv <= kMaxRep;
}

// The workspace: kAttnCounters arrival counters (zero when allocated, left zero by every
// launch), then the split partials.
hipError_t launch_attention(const float* q, const float* kc, const float* vc, int rows, int pos0,
                            int n_head, int n_kv, int head_dim, float* out, void* ws,
                            size_t ws_bytes, hipStream_t stream, float rope_base) {
    if (rows <= 0) return hipSuccess;
    if (!attention_supported(head_dim, n_head, n_kv)) return hipErrorInvalidValue;
    if (rope_base > 0.0f && rows != 1) return hipErrorInvalidValue;
    if (rope_base <= 0.0f && attention_uses_mfma(rows, pos0, n_head, n_kv, head_dim)) {
        switch (head_dim) {
            case 64: return launch_attention_mfma_hd<64, 2, 8>(q, kc, vc, rows, pos0, n_head, n_kv, out, stream);
            case 128: return launch_attention_mfma_hd<128, 2, 8>(q, kc, vc, rows, pos0, n_head, n_kv, out, stream);
            default: return launch_attention_mfma_hd<256, 1, 4>(q, kc, vc, rows, pos0, n_head, n_kv, out, stream);
        }
    }
    float* k_new = rope_base > 0.0f ? const_cast<float*>(kc) + (size_t)pos0 * n_kv * head_dim : nullptr;
    constexpr size_t kCountBytes = kAttnCounters * sizeof(int);
    int* counters = ws && ws_bytes > kCountBytes ? (int*)ws : nullptr;
    float* part = counters ? (float*)((char*)ws + kCountBytes) : nullptr;
    const size_t part_floats = counters ? (ws_bytes - kCountBytes) / sizeof(float) : 0;
    switch (head_dim) {
        case 64: return launch_attention_hd<64>(q, kc, vc, rows, pos0, n_head, n_kv, out, part, part_floats, counters, rope_base, k_new, stream);
        case 128: return launch_attention_hd<128>(q, kc, vc, rows, pos0, n_head, n_kv, out, part, part_floats, counters, rope_base, k_new, stream);
        default: return launch_attention_hd<256>(q, kc, vc, rows, pos0, n_head, n_kv, out, part, part_floats, counters, rope_base, k_new, stream);
    }
}

}  // namespace cllm_hip
