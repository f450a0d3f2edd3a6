// float_units.h -- decoding of 32-element units of weight rows to fp32 on the device: the
// float-dot kernels (k_gemv_f.hip, k_gemm_f.hip) and the row and span dequantization.
#pragma once

#include "device_utils.h"
#include "ggml_blocks.h"

namespace cllm_hip {

// byte b (0..3) of dword v as a float: v_cvt_f32_ubyte{0..3}
__device__ __forceinline__ float ubyte_f(uint32_t v, int b) {
    return (float)((v >> (8 * b)) & 0xFFu);
}

// The 16 codes held in the bytes of v[0..3] (element order; unsigned, or int8 when SIGNED) as
// floats. The words pass through an empty asm first: the compiler knows which bits the
// callers' masks clear and would otherwise turn each byte into a narrower bit-field extract
// plus v_cvt_f32_ubyte0, instead of one v_cvt_f32_ubyte{0..3}.
template <bool SIGNED>
__device__ __forceinline__ void codes16(const uint32_t (&v)[4], float (&c)[16]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t w = v[i];
        asm volatile("" : "+v"(w));
#pragma unroll
        for (int b = 0; b < 4; ++b)
            c[4 * i + b] = SIGNED ? (float)(int8_t)((w >> (8 * b)) & 0xFFu) : ubyte_f(w, b);
    }
}

// sum over 16 elements of x[e] * c[e], x 16 consecutive floats (16-byte aligned), in order
__device__ __forceinline__ float dot16(const float (&c)[16], const float* x) {
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float4 xv = *(const float4*)(x + 4 * i);
        s = __builtin_fmaf(xv.x, c[4 * i], s);
        s = __builtin_fmaf(xv.y, c[4 * i + 1], s);
        s = __builtin_fmaf(xv.z, c[4 * i + 2], s);
        s = __builtin_fmaf(xv.w, c[4 * i + 3], s);
    }
    return s;
}

// bits 0..3 of h (h < 16) to bit 4 of bytes 0..3: h * 0x204081 puts bit j at bit 8 j
__device__ __forceinline__ uint32_t spread4_bit4(uint32_t h) {
    return ((h * 0x00204081u) & 0x01010101u) << 4;
}

// ------------------------------------------------------------------------- unit decoders
// Each FUnit<T> loads the raw bytes of unit u of a row (load) and turns them into the 32
// fp32 weights of that unit, in element order (decode).

template <uint32_t T> struct FUnit;

// F32: 128 bytes (quant.cpp:29-31)
template <> struct FUnit<T_F32> {
    struct Raw { u32x4 v[8]; };
    __device__ __forceinline__ static Raw load(const uint8_t* row, int u) {
        Raw r;
        const u32x4* p = (const u32x4*)(row + (size_t)u * 128);
#pragma unroll
        for (int i = 0; i < 8; ++i) r.v[i] = p[i];
        return r;
    }
    __device__ __forceinline__ static void decode(const Raw& r, int, float (&w)[32]) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            // element values are copied out first: __builtin_bit_cast applied to a vector
            // element expression reads element 0 with this compiler
            const uint32_t e[4] = {r.v[i].x, r.v[i].y, r.v[i].z, r.v[i].w};
#pragma unroll
            for (int c = 0; c < 4; ++c) w[4 * i + c] = __builtin_bit_cast(float, e[c]);
        }
    }
};

// F16: 64 bytes, exact conversion (quant.cpp:34-37)
template <> struct FUnit<T_F16> {
    struct Raw { u32x4 v[4]; };
    __device__ __forceinline__ static Raw load(const uint8_t* row, int u) {
        Raw r;
        const u32x4* p = (const u32x4*)(row + (size_t)u * 64);
#pragma unroll
        for (int i = 0; i < 4; ++i) r.v[i] = p[i];
        return r;
    }
    __device__ __forceinline__ static void decode(const Raw& r, int, float (&w)[32]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t d[4] = {r.v[i].x, r.v[i].y, r.v[i].z, r.v[i].w};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                w[8 * i + 2 * k] = f16_to_f32(d[k] & 0xFFFFu);
                w[8 * i + 2 * k + 1] = f16_to_f32(d[k] >> 16);
            }
        }
    }
};

// Q8_1: [d f16][s f16][qs i8 x32], 36 bytes, value d * q; s is not used (quant.cpp:203-214)
template <> struct FUnit<T_Q8_1> {
    struct Raw { u32x4_a4 a, b; uint32_t c; };
    __device__ __forceinline__ static Raw load(const uint8_t* row, int u) {
        const uint8_t* p = row + (size_t)u * 36;
        Raw r;
        r.a = *(const u32x4_a4*)p;
        r.b = *(const u32x4_a4*)(p + 16);
        r.c = *(const uint32_t*)(p + 32);
        return r;
    }
    __device__ __forceinline__ static void decode(const Raw& r, int, float (&w)[32]) {
        const float d = f16_to_f32(r.a.x & 0xFFFFu);
        const uint32_t q[8] = {r.a.y, r.a.z, r.a.w, r.b.x, r.b.y, r.b.z, r.b.w, r.c};
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int b = 0; b < 4; ++b)
                w[4 * i + b] = d * (float)(int8_t)((q[i] >> (8 * b)) & 0xFFu);
    }
    // w = d q: A = d, no offset
    template <int MR>
    __device__ __forceinline__ static void gdot(const Raw& r, int, const float* xp, int xstride,
                                                const float*, int, float (&acc)[MR]) {
        const float d = f16_to_f32(r.a.x & 0xFFFFu);
        const uint32_t q0[4] = {r.a.y, r.a.z, r.a.w, r.b.x}, q1[4] = {r.b.y, r.b.z, r.b.w, r.c};
        float c0[16], c1[16];
        codes16<true>(q0, c0);
        codes16<true>(q1, c1);
#pragma unroll
        for (int t = 0; t < MR; ++t) {
            const float* xt = xp + (size_t)t * xstride;
            acc[t] = __builtin_fmaf(d, dot16(c0, xt) + dot16(c1, xt + 16), acc[t]);
        }
    }
};

// Q4_1: [d][m][qs 16 B], 20 bytes; byte j: low nibble = element j, high = element j + 16;
// value d * q + m (quant.cpp:164-177)
template <> struct FUnit<T_Q4_1> {
    struct Raw { uint32_t dm; u32x4_a4 qs; };
    __device__ __forceinline__ static Raw load(const uint8_t* row, int u) {
        const uint8_t* p = row + (size_t)u * 20;
        Raw r;
        r.dm = *(const uint32_t*)p;
        r.qs = *(const u32x4_a4*)(p + 4);
        return r;
    }
    __device__ __forceinline__ static void decode(const Raw& r, int, float (&w)[32]) {
        const float d = f16_to_f32(r.dm & 0xFFFFu), m = f16_to_f32(r.dm >> 16);
        const uint32_t q[4] = {r.qs.x, r.qs.y, r.qs.z, r.qs.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t lo = q[i] & 0x0F0F0F0Fu, hi = (q[i] >> 4) & 0x0F0F0F0Fu;
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                w[4 * i + b] = __builtin_fmaf(d, ubyte_f(lo, b), m);
                w[16 + 4 * i + b] = __builtin_fmaf(d, ubyte_f(hi, b), m);
            }
        }
    }
    // w = d q + m over the 32 elements: A = d, B = m
    template <int MR>
    __device__ __forceinline__ static void gdot(const Raw& r, int, const float* xp, int xstride,
                                                const float* xg, int gstride, float (&acc)[MR]) {
        const float d = f16_to_f32(r.dm & 0xFFFFu), m = f16_to_f32(r.dm >> 16);
        const uint32_t q[4] = {r.qs.x, r.qs.y, r.qs.z, r.qs.w};
        uint32_t lo[4], hi[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            lo[i] = q[i] & 0x0F0F0F0Fu;
            hi[i] = (q[i] >> 4) & 0x0F0F0F0Fu;
        }
        float c0[16], c1[16];
        codes16<false>(lo, c0);
        codes16<false>(hi, c1);
#pragma unroll
        for (int t = 0; t < MR; ++t) {
            const float* xt = xp + (size_t)t * xstride;
            const float s = dot16(c0, xt) + dot16(c1, xt + 16);
            const float xsum = xg[(size_t)t * gstride] + xg[(size_t)t * gstride + 1];
            acc[t] = __builtin_fmaf(m, xsum, __builtin_fmaf(d, s, acc[t]));
        }
    }
};

// Q5_1: [d][m][qh u32][qs 16 B], 24 bytes; bit j of qh is bit 4 of element j
// (quant.cpp:182-200)
template <> struct FUnit<T_Q5_1> {
    struct Raw { u32x2_a4 dmh; u32x4_a4 qs; };
    __device__ __forceinline__ static Raw load(const uint8_t* row, int u) {
        const uint8_t* p = row + (size_t)u * 24;
        Raw r;
        r.dmh = *(const u32x2_a4*)p;
        r.qs = *(const u32x4_a4*)(p + 8);
        return r;
    }
    __device__ __forceinline__ static void decode(const Raw& r, int, float (&w)[32]) {
        const float d = f16_to_f32(r.dmh.x & 0xFFFFu), m = f16_to_f32(r.dmh.x >> 16);
        const uint32_t qh = r.dmh.y;
        const uint32_t q[4] = {r.qs.x, r.qs.y, r.qs.z, r.qs.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            // bit 4 of elements 4i..4i+3 and 16+4i..: qh bits 4i.. and 16+4i.. moved to bit 4
            // of each byte
            const uint32_t h0 = (qh >> (4 * i)) & 0xFu, h1 = (qh >> (16 + 4 * i)) & 0xFu;
            const uint32_t s0 = ((h0 & 1u) | ((h0 & 2u) << 7) | ((h0 & 4u) << 14) | ((h0 & 8u) << 21)) << 4;
            const uint32_t s1 = ((h1 & 1u) | ((h1 & 2u) << 7) | ((h1 & 4u) << 14) | ((h1 & 8u) << 21)) << 4;
            const uint32_t lo = (q[i] & 0x0F0F0F0Fu) | s0, hi = ((q[i] >> 4) & 0x0F0F0F0Fu) | s1;
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                w[4 * i + b] = __builtin_fmaf(d, ubyte_f(lo, b), m);
                w[16 + 4 * i + b] = __builtin_fmaf(d, ubyte_f(hi, b), m);
            }
        }
    }
    // w = d q + m over the 32 elements (q 5 bits): A = d, B = m
    template <int MR>
    __device__ __forceinline__ static void gdot(const Raw& r, int, const float* xp, int xstride,
                                                const float* xg, int gstride, float (&acc)[MR]) {
        const float d = f16_to_f32(r.dmh.x & 0xFFFFu), m = f16_to_f32(r.dmh.x >> 16);
        const uint32_t qh = r.dmh.y;
        const uint32_t q[4] = {r.qs.x, r.qs.y, r.qs.z, r.qs.w};
        uint32_t lo[4], hi[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            lo[i] = (q[i] & 0x0F0F0F0Fu) | spread4_bit4((qh >> (4 * i)) & 0xFu);
            hi[i] = ((q[i] >> 4) & 0x0F0F0F0Fu) | spread4_bit4((qh >> (16 + 4 * i)) & 0xFu);
        }
        float c0[16], c1[16];
        codes16<false>(lo, c0);
        codes16<false>(hi, c1);
#pragma unroll
        for (int t = 0; t < MR; ++t) {
            const float* xt = xp + (size_t)t * xstride;
            const float s = dot16(c0, xt) + dot16(c1, xt + 16);
            const float xsum = xg[(size_t)t * gstride] + xg[(size_t)t * gstride + 1];
            acc[t] = __builtin_fmaf(m, xsum, __builtin_fmaf(d, s, acc[t]));
        }
    }
};

// Q2_K: [scales 16][qs 64][d][dmin], 84 bytes. Unit v = 4 h + j of a super-block: elements
// 32 v + l take bits 2j..2j+1 of qs[32 h + l], with scale byte 8 h + 2 j for l < 16 and
// 8 h + 2 j + 1 for l >= 16 (low nibble scale, high nibble min); value
// d * sc * q - dmin * m (quant.cpp:218-248).
template <> struct FUnit<T_Q2_K> {
    struct Raw { u32x4_a4 q0, q1; uint32_t sc; uint32_t dd; };
    __device__ __forceinline__ static Raw load(const uint8_t* row, int u) {
        const uint8_t* blk = row + (size_t)(u >> 3) * 84;
        const int v = u & 7, h = v >> 2, j = v & 3;
        Raw r;
        r.q0 = *(const u32x4_a4*)(blk + 16 + 32 * h);
        r.q1 = *(const u32x4_a4*)(blk + 32 + 32 * h);
        r.sc = ld_u16(blk + 8 * h + 2 * j);
        r.dd = *(const uint32_t*)(blk + 80);
        return r;
    }
    __device__ __forceinline__ static void decode(const Raw& r, int u, float (&w)[32]) {
        const int sh = 2 * (u & 3);
        const float d = f16_to_f32(r.dd & 0xFFFFu), dmin = f16_to_f32(r.dd >> 16);
        const uint32_t q[8] = {r.q0.x, r.q0.y, r.q0.z, r.q0.w, r.q1.x, r.q1.y, r.q1.z, r.q1.w};
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            const uint32_t scb = (r.sc >> (8 * g)) & 0xFFu;
            const float dl = d * (float)(scb & 0xFu), ml = dmin * (float)(scb >> 4);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t v = (q[4 * g + i] >> sh) & 0x03030303u;
#pragma unroll
                for (int b = 0; b < 4; ++b) w[16 * g + 4 * i + b] = __builtin_fmaf(dl, ubyte_f(v, b), -ml);
            }
        }
    }
};

// Q3_K: [hmask 32][qs 64][scales 12][d], 110 bytes (2-byte aligned blocks). Unit v = 4 h + j:
// elements 32 v + l take bits 2j..2j+1 of qs[32 h + l] minus 4 unless bit 4h + j of
// hmask[l] is set, with the signed 6-bit scale 8 h + 2 j (l < 16) or 8 h + 2 j + 1 (l >= 16);
// value d * (scale - 32) * q (quant.cpp:252-298).
template <> struct FUnit<T_Q3_K> {
    struct Raw { uint32_t hm[8], q[8], sc[3], d; };
    __device__ __forceinline__ static Raw load(const uint8_t* row, int u) {
        const uint8_t* blk = row + (size_t)(u >> 3) * 110;
        const int h = (u & 7) >> 2;
        Raw r;
        ld_a2<8>(blk, r.hm);
        ld_a2<8>(blk + 32 + 32 * h, r.q);
        ld_a2<3>(blk + 96, r.sc);
        r.d = ld_u16(blk + 108);
        return r;
    }
    // Scale i (0..15) of the 12 packed bytes b (as dwords s[0..2]): low four bits from byte
    // i (i < 8, low nibble) or byte i - 8 (i >= 8, high nibble), top two bits from byte
    // 8 + i % 4 at bit 2 (i / 4) (the aux shuffle of quant.cpp:259-265).
    __device__ __forceinline__ static int scale(const uint32_t (&s)[3], int i) {
        const int grp = i >> 2, ii = i & 3;
        // bytes 0-7 as one 64-bit value, shifted (an indexed pick of s[0] / s[1] would be
        // lowered to a scratch-memory load)
        const uint64_t s01 = (uint64_t)s[0] | ((uint64_t)s[1] << 32);
        const uint32_t src = (uint32_t)(s01 >> (32 * (grp & 1) + 8 * ii));
        const uint32_t lo = (grp < 2 ? src : src >> 4) & 0xFu;
        const uint32_t hi = (s[2] >> (8 * ii + 2 * grp)) & 3u;
        return (int)(lo | (hi << 4)) - 32;
    }
    __device__ __forceinline__ static void decode(const Raw& r, int u, float (&w)[32]) {
        const int v = u & 7, h = v >> 2, j = v & 3;
        const float d = f16_to_f32(r.d);
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            const float dl = d * (float)scale(r.sc, 8 * h + 2 * j + g);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                // q2 | hbit << 2 per byte, so value = byte - 4
                const uint32_t q2 = (r.q[4 * g + i] >> (2 * j)) & 0x03030303u;
                const uint32_t hb = ((r.hm[4 * g + i] >> (4 * h + j)) & 0x01010101u) << 2;
                const uint32_t qv = q2 | hb;
#pragma unroll
                for (int b = 0; b < 4; ++b) w[16 * g + 4 * i + b] = dl * (ubyte_f(qv, b) - 4.0f);
            }
        }
    }
};

// The six vec_dot types, for the row dequantization below (the GEMV keeps their integer
// kernels). Values as the reference's deq_* produce them (quant.cpp:39-161, 302-336).

// Q8_0: [d][qs i8 x32], 34 bytes (2-byte aligned blocks): d * q
template <> struct FUnit<T_Q8_0> {
    struct Raw { uint32_t d; uint32_t q[8]; };
    __device__ __forceinline__ static Raw load(const uint8_t* row, int u) {
        const uint8_t* blk = row + (size_t)u * 34;
        Raw r;
        r.d = ld_u16(blk);
        ld_a2<8>(blk + 2, r.q);
        return r;
    }
    __device__ __forceinline__ static void decode(const Raw& r, int, float (&w)[32]) {
        const float d = f16_to_f32(r.d);
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int b = 0; b < 4; ++b) w[4 * i + b] = d * (float)(int8_t)((r.q[i] >> (8 * b)) & 0xFFu);
    }
};

// Q4_0: [d][qs 16 B], 18 bytes: d * (q - 8), low nibble element j, high nibble j + 16
template <> struct FUnit<T_Q4_0> {
    struct Raw { uint32_t d; uint32_t q[4]; };
    __device__ __forceinline__ static Raw load(const uint8_t* row, int u) {
        const uint8_t* blk = row + (size_t)u * 18;
        Raw r;
        r.d = ld_u16(blk);
        ld_a2<4>(blk + 2, r.q);
        return r;
    }
    __device__ __forceinline__ static void decode(const Raw& r, int, float (&w)[32]) {
        const float d = f16_to_f32(r.d);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t lo = r.q[i] & 0x0F0F0F0Fu, hi = (r.q[i] >> 4) & 0x0F0F0F0Fu;
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                w[4 * i + b] = d * (ubyte_f(lo, b) - 8.0f);
                w[16 + 4 * i + b] = d * (ubyte_f(hi, b) - 8.0f);
            }
        }
    }
};

// Q5_0: [d][qh u32][qs 16 B], 22 bytes: d * (q - 16), bit j of qh = bit 4 of element j
template <> struct FUnit<T_Q5_0> {
    struct Raw { uint32_t d; uint32_t qh[1]; uint32_t q[4]; };
    __device__ __forceinline__ static Raw load(const uint8_t* row, int u) {
        const uint8_t* blk = row + (size_t)u * 22;
        Raw r;
        r.d = ld_u16(blk);
        ld_a2<1>(blk + 2, r.qh);
        ld_a2<4>(blk + 6, r.q);
        return r;
    }
    __device__ __forceinline__ static void decode(const Raw& r, int, float (&w)[32]) {
        const float d = f16_to_f32(r.d);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const int j = 4 * i + b;
                const uint32_t byte = (r.q[i] >> (8 * b)) & 0xFFu;
                const uint32_t q0 = (byte & 0xFu) | (((r.qh[0] >> j) & 1u) << 4);
                const uint32_t q1 = (byte >> 4) | (((r.qh[0] >> (j + 16)) & 1u) << 4);
                w[j] = d * ((float)q0 - 16.0f);
                w[j + 16] = d * ((float)q1 - 16.0f);
            }
        }
    }
};

// Q4_K / Q5_K: unit u = sub-block u of the super-block: low (u even) or high (u odd)
// nibbles of the 32-byte chunk u / 2, Q5_K adding bit u of qh[l] as bit 4; value
// d * sc_u * q - dmin * m_u (quant.cpp:82-108, 302-336).
template <bool Q5>
struct FUnitK45 {
    struct Raw { uint32_t dd; uint32_t s[3]; u32x4 q0, q1, h0, h1; };
    __device__ __forceinline__ static Raw load(const uint8_t* row, int u) {
        const uint8_t* blk = row + (size_t)(u >> 3) * (Q5 ? 176 : 144);
        const int c = (u & 7) >> 1;
        Raw r;
        r.dd = *(const uint32_t*)blk;
        r.s[0] = *(const uint32_t*)(blk + 4);
        r.s[1] = *(const uint32_t*)(blk + 8);
        r.s[2] = *(const uint32_t*)(blk + 12);
        const u32x4* qs = (const u32x4*)(blk + (Q5 ? 48 : 16) + 32 * c);
        r.q0 = qs[0];
        r.q1 = qs[1];
        if constexpr (Q5) {
            r.h0 = *(const u32x4*)(blk + 16);
            r.h1 = *(const u32x4*)(blk + 32);
        }
        return r;
    }
    __device__ __forceinline__ static void decode(const Raw& r, int u, float (&w)[32]) {
        const int k = u & 7;
        int sc, m;
        k4_scale_min(r.s[0], r.s[1], r.s[2], k, sc, m);
        const float d1 = f16_to_f32(r.dd & 0xFFFFu) * (float)sc;
        const float m1 = f16_to_f32(r.dd >> 16) * (float)m;
        const uint32_t q[8] = {r.q0.x, r.q0.y, r.q0.z, r.q0.w, r.q1.x, r.q1.y, r.q1.z, r.q1.w};
        const uint32_t h[8] = {r.h0.x, r.h0.y, r.h0.z, r.h0.w, r.h1.x, r.h1.y, r.h1.z, r.h1.w};
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            uint32_t v = (k & 1) ? (q[i] >> 4) & 0x0F0F0F0Fu : q[i] & 0x0F0F0F0Fu;
            if constexpr (Q5) v |= ((h[i] >> k) & 0x01010101u) << 4;
#pragma unroll
            for (int b = 0; b < 4; ++b) w[4 * i + b] = __builtin_fmaf(d1, ubyte_f(v, b), -m1);
        }
    }
};
template <> struct FUnit<T_Q4_K> : FUnitK45<false> {};
template <> struct FUnit<T_Q5_K> : FUnitK45<true> {};

// Q6_K: [ql 128][qh 64][sc i8 x16][d], 210 bytes (2-byte aligned). Unit u = 4 g + i (half g,
// quarter i): element l takes the low (i < 2) or high nibble of ql[64 g + 32 (i & 1) + l],
// bits 2i..2i+1 of qh[32 g + l] as bits 4-5, scale sc[8 g + 2 i + l / 16]; value
// d * sc * (q - 32) (quant.cpp:135-161).
template <> struct FUnit<T_Q6_K> {
    struct Raw { uint32_t ql[8], qh[8], sc, d; };
    __device__ __forceinline__ static Raw load(const uint8_t* row, int u) {
        const uint8_t* blk = row + (size_t)(u >> 3) * 210;
        const int g = (u & 7) >> 2, i = u & 3;
        Raw r;
        ld_a2<8>(blk + 64 * g + 32 * (i & 1), r.ql);
        ld_a2<8>(blk + 128 + 32 * g, r.qh);
        r.sc = ld_u16(blk + 192 + 8 * g + 2 * i);
        r.d = ld_u16(blk + 208);
        return r;
    }
    __device__ __forceinline__ static void decode(const Raw& r, int u, float (&w)[32]) {
        const int i = u & 3;
        const float d = f16_to_f32(r.d);
#pragma unroll
        for (int hb = 0; hb < 2; ++hb) {
            const float ds = d * (float)(int8_t)((r.sc >> (8 * hb)) & 0xFFu);  // exact
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t lo = (i < 2 ? r.ql[4 * hb + j] : r.ql[4 * hb + j] >> 4) & 0x0F0F0F0Fu;
                const uint32_t hi = ((r.qh[4 * hb + j] >> (2 * i)) & 0x03030303u) << 4;
                const uint32_t v = lo | hi;
#pragma unroll
                for (int b = 0; b < 4; ++b) w[16 * hb + 4 * j + b] = ds * (ubyte_f(v, b) - 32.0f);
            }
        }
    }
};

}  // namespace cllm_hip
