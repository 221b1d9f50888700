/*
 * The cache append's row math, shared by the append kernels (kv_append.hip) and the fused decode step
 * (attention.hip), so both produce the same bits: one (token, head) row per wave, lane l holding the rotation
 * pair (dims l, l + 64). Reference row math: model/kernels/qk_row.cuh:19-51 (qk_row_sum, qk_rstd, qk_rotate) and
 * model/kernels/decode.cu:481-494 (the value-embedding gate); the summation order is fixed here (lane partial
 * x[l]^2 + x[l+64]^2, then the xor butterfly over offsets 32..1) and 1/sqrt is correctly rounded where the
 * reference has rsqrtf. The value-embedding gate's exponential is exp_rn (below) where the reference has expf, so
 * the gate's bits follow from its fixed fp32 order alone.
 */
#pragma once

#include "nc_device.h"

namespace nc {

/* RMS norm (eps FLT_EPSILON), gain and -theta rotation of one row held as lane pairs (x1 = dim l,
 * x2 = dim l + 64); results before the bf16 rounding. Every operation is a single rounded fp32 op in the
 * order of the oracle's qk_norm_rope. All 64 lanes of the wave must call it together. */
__device__ __forceinline__ void norm_rope_pair(float x1, float x2, float g1, float g2, float c, float s, float &y1,
                                               float &y2) {
    const float part = x1 * x1 + x2 * x2;
    const float ss = wave_sum_butterfly(part);
    const float v = ss / 128.0f + FLT_EPS;
    const float r = 1.0f / __builtin_sqrtf(v);  /* correctly rounded (HIP's __fsqrt_rn is not, here) */
    const float n1 = (x1 * r) * g1;
    const float n2 = (x2 * r) * g2;
    y1 = n1 * c + n2 * s;
    y2 = n2 * c - n1 * s;
}

/* The code e4m3_encode(clamp(x / scale, +-448)) of a bf16 value x of a row whose scale is amax / 448 (|x| <= amax).
 * For scale >= 2^-80 (fast) the division becomes a product with r = 1 / scale (correctly rounded) and one FMA
 * correction of |x| (Markstein), the sign copied from x: every finite bf16 x with |x| <= amax, against every bf16
 * amax, gives the same code this way as by the division (an exhaustive check, tests/quant_division_check.c). Smaller
 * scales divide. */
__device__ __forceinline__ uint32_t quant_code(float x, float scale, float r, bool fast) {
    if (!fast) return e4m3_encode(fminf(fmaxf(x / scale, -FP8_MAX), FP8_MAX));
    const float ax = fabsf(x);
    const float q0 = ax * r;
    const float q = __builtin_fmaf(__builtin_fmaf(-q0, scale, ax), r, q0);
    return e4m3_encode(fminf(q, FP8_MAX)) | ((__float_as_uint(x) >> 24) & 0x80u);
}

constexpr float QUANT_FAST_SCALE = 0x1p-80f;   /* quant_code's fast path: scales from here up */

/* Absmax e4m3fn quantization of one row (lane pair x1 = dim l, x2 = dim l + 64, bf16 values): the row's scale
 * amax / 448 (1 for an all-zero row), returned in every lane, and this lane's two codes. */
__device__ __forceinline__ float quantize_pair(float x1, float x2, uint32_t &c1, uint32_t &c2) {
    const float amax = wave_max(fmaxf(fabsf(x1), fabsf(x2)));
    const float scale = amax > 0.0f ? amax / FP8_MAX : 1.0f;
    const bool fast = scale >= QUANT_FAST_SCALE;
    const float r = 1.0f / scale;
    c1 = quant_code(x1, scale, r, fast);
    c2 = quant_code(x2, scale, r, fast);
    return scale;
}

/* e^x of an fp32 x, rounded once to fp32: the double exponential (within an ulp of double precision) rounded to
 * float. This is the correctly rounded e^x except where e^x lies within about 2^-52 (relative) of the midpoint of two
 * floats, so it does not depend on a float exponential's own error. */
__device__ __forceinline__ float exp_rn(float x) { return (float)exp((double)x); }

/* Value-embedding mix of one value row: g = 2 sigmoid(w . h) from the token's normed stream h (C wide, lane-strided
 * FMAs, then the butterfly) and v = bf16(v + g e) with e the token's embedding row for this head. */
__device__ __forceinline__ void ve_mix_pair(const uint16_t *h, const float *w, int C, const uint16_t *e, int lane,
                                            float &v1, float &v2) {
    float d = 0.0f;
    for (int i = lane; i < C; i += WAVE) d = __builtin_fmaf(bf16_to_f32(h[i]), w[i], d);
    d = wave_sum_butterfly(d);
    const float g = 2.0f * (1.0f / (1.0f + exp_rn(-d)));
    v1 = bf16_to_f32(f32_to_bf16(v1 + g * bf16_to_f32(e[lane])));
    v2 = bf16_to_f32(f32_to_bf16(v2 + g * bf16_to_f32(e[lane + HALF])));
}

/* The same row math with 16 lanes a row, four rows a wave: lane i of a 16-lane group holds dims 4 i .. 4 i + 3 (elements
 * 0 .. 3) and 64 + 4 i .. 64 + 4 i + 3 (elements 4 .. 7) of its row, so a row moves by two 8-byte accesses a lane and its
 * rotation pairs (elements j, j + 4) are lane-local. Pair j of lane i stands for lane l = 4 i + j of the one-row-a-wave
 * form: its butterfly steps 32, 16, 8 and 4 pair lanes i with i ^ 8, i ^ 4, i ^ 2 and i ^ 1, and steps 2 and 1 pair
 * elements, so every sum is formed in the same order and has the same bits. All 16 lanes of a group must call these
 * together. (Eight consecutive dims a lane, by 16-byte accesses, spread the order's first steps over eight values a lane
 * and the pairs over lanes: the append of 8 x 512
 * tokens took 15 us that way, 12.8 this way.) */
__device__ __forceinline__ float lane16_sum(float (&d)[4]) {
#pragma unroll
    for (int j = 0; j < 4; j++) d[j] = d[j] + lane_xor_dpp<8>(d[j]);
#pragma unroll
    for (int j = 0; j < 4; j++) d[j] = d[j] + lane_xor_dpp<4>(d[j]);
#pragma unroll
    for (int j = 0; j < 4; j++) d[j] = d[j] + lane_xor_dpp<2>(d[j]);
#pragma unroll
    for (int j = 0; j < 4; j++) d[j] = d[j] + lane_xor_dpp<1>(d[j]);
    return (d[0] + d[2]) + (d[1] + d[3]);
}

/* 1 / sqrt(mean x^2 + FLT_EPSILON) of the row, as norm_rope_pair's r. */
__device__ __forceinline__ float rstd16(const float (&x)[8]) {
    float part[4];
#pragma unroll
    for (int j = 0; j < 4; j++) part[j] = x[j] * x[j] + x[j + 4] * x[j + 4];
    const float v = lane16_sum(part) / 128.0f + FLT_EPS;
    return 1.0f / __builtin_sqrtf(v);
}

/* norm_rope_pair in this form. g: the lane's gains; c, s: cos and sin of its four pairs. */
__device__ __forceinline__ void norm_rope16(const float (&x)[8], const float (&g)[8], const float (&c)[4],
                                            const float (&s)[4], float (&y)[8]) {
    const float r = rstd16(x);
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const float n1 = (x[j] * r) * g[j];
        const float n2 = (x[j + 4] * r) * g[j + 4];
        y[j] = n1 * c[j] + n2 * s[j];
        y[j + 4] = n2 * c[j] - n1 * s[j];
    }
}

/* A lane's elements of a row at any element alignment (the declared alignment is the element's). */
typedef uint32_t u32x2_a2 __attribute__((ext_vector_type(2), aligned(2)));
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ uint4 load_row16(const uint16_t *row, int i) {
    const u32x2_a2 a = *reinterpret_cast<const u32x2_a2 *>(row + 4 * i);
    const u32x2_a2 b = *reinterpret_cast<const u32x2_a2 *>(row + HALF + 4 * i);
    return uint4{a[0], a[1], b[0], b[1]};
}

__device__ __forceinline__ void unpack8(const uint4 &r, float (&x)[8]) {
    const uint32_t u[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int k = 0; k < 4; k++) {
        x[2 * k] = __uint_as_float(u[k] << 16);
        x[2 * k + 1] = __uint_as_float(u[k] & 0xFFFF0000u);
    }
}

__device__ __forceinline__ void load4_f32(const float *p, float (&x)[4]) {
    const u32x4_a4 a = *reinterpret_cast<const u32x4_a4 *>(p);
#pragma unroll
    for (int k = 0; k < 4; k++) x[k] = __uint_as_float(a[k]);
}

/* fp32 [128] (a gain) as a lane's elements. */
__device__ __forceinline__ void load_gain16(const float *g, int i, float (&x)[8]) {
    float a[4], b[4];
    load4_f32(g + 4 * i, a);
    load4_f32(g + HALF + 4 * i, b);
#pragma unroll
    for (int k = 0; k < 4; k++) {
        x[k] = a[k];
        x[4 + k] = b[k];
    }
}

/* Rounded to bf16 (nearest even, v_cvt_pk_bf16_f32), packed. */
__device__ __forceinline__ uint4 pack8(const float (&x)[8]) {
    bf16x8 v;
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = (__bf16)x[e];
    return __builtin_bit_cast(uint4, v);
}

__device__ __forceinline__ void store_row16(uint16_t *row, int i, const float (&x)[8]) {
    const uint4 u = pack8(x);
    *reinterpret_cast<u32x2_a2 *>(row + 4 * i) = u32x2_a2{u.x, u.y};
    *reinterpret_cast<u32x2_a2 *>(row + HALF + 4 * i) = u32x2_a2{u.z, u.w};
}

/* quantize_pair in this form: the row's scale, and the lane's codes of its two runs of four dims, packed. */
__device__ __forceinline__ float quantize16(const float (&x)[8], uint32_t (&code)[2]) {
    float m = fabsf(x[0]);
#pragma unroll
    for (int e = 1; e < 8; e++) m = fmaxf(m, fabsf(x[e]));
    m = fmaxf(m, lane_xor_dpp<8>(m));
    m = fmaxf(m, lane_xor_dpp<4>(m));
    m = fmaxf(m, lane_xor_dpp<2>(m));
    const float amax = fmaxf(m, lane_xor_dpp<1>(m));
    const float scale = amax > 0.0f ? amax / FP8_MAX : 1.0f;
    const bool fast = scale >= QUANT_FAST_SCALE;
    const float r = 1.0f / scale;
    code[0] = code[1] = 0u;
#pragma unroll
    for (int e = 0; e < 8; e++) code[e >> 2] |= quant_code(x[e], scale, r, fast) << (8 * (e & 3));
    return scale;
}

/* ve_mix_pair in this form: the gate's 64 FMA chains (chain l: elements l, l + 64, ...) run four a lane, lane i chains
 * 4 i .. 4 i + 3, so h and w move by 8- and 16-byte loads. */
__device__ __forceinline__ void ve_mix16(const uint16_t *h, const float *w, int C, const uint16_t *e, int i,
                                         float (&v)[8]) {
    const uint4 emb = load_row16(e, i);
    float d[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    const int whole = C / WAVE * WAVE;
#pragma unroll 4
    for (int k = 4 * i; k < whole; k += WAVE) {
        const u32x2_a2 x = *reinterpret_cast<const u32x2_a2 *>(h + k);
        float y[4];
        load4_f32(w + k, y);
#pragma unroll
        for (int j = 0; j < 4; j++)
            d[j] = __builtin_fmaf(__uint_as_float(j & 1 ? x[j >> 1] & 0xFFFF0000u : x[j >> 1] << 16), y[j], d[j]);
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int k = whole + 4 * i + j;
        if (k < C) d[j] = __builtin_fmaf(bf16_to_f32(h[k]), w[k], d[j]);
    }
    const float g = 2.0f * (1.0f / (1.0f + exp_rn(-lane16_sum(d))));
    float ev[8];
    unpack8(emb, ev);
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] = v[j] + g * ev[j];
    unpack8(pack8(v), v);
}

}  // namespace nc
