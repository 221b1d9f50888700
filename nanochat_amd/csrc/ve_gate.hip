/*
 * Value-embedding gate and mix of training, gfx950: the reference's model/kernels/ve_gate.cu (called through
 * model/ops/ve_gate.py by model/ops/flash_attn.py:340 and :391).
 *
 * Forward, per row r of the normed stream n (rows = B*T, C = 128 H for H heads):
 *   z[h]       = sum_c n[r][c] w[h][c]                           fp32 fused multiply-adds, then a wave reduction
 *   gate[r][h] = 2 * (1 / (1 + exp(-z[h])))                      fp32
 *   out[r][c]  = bf16(v[r][c] + gate[r][c / 128] * bf16(table[idx[r]][c]))   product and sum each rounded once
 * Backward, per row r, visited in token order (position p holds row order[p] and token ids[p]):
 *   dg[h]        = sum over head h's 128 columns of dout[r][c] * bf16(table[t][c])
 *   dz[r][h]     = bf16(2 dg[h] (1 - s) s) with s = gate[r][h] / 2   (dz_fp32, unrounded, feeds dn)
 *   dn[r][c]     = bf16(sum_h dz_fp32[h] w[h][c])
 *   dtable[t][c] += sum over the rows of token t of bf16(gate[r][c / 128] * dout[r][c])   (fp32, added in)
 * dw = dz^T n (nc_ve_weight_grad; a GEMM on the host side in the reference). ids must hold equal tokens adjacently (sorted,
 * the reference's contract, model/ops/ve_gate.py:23-26): the table gradient of a token split into separate runs is
 * undefined.
 *
 * Mapping: one wave per row. Lane l holds the 8-column chunks c = (i*64 + l)*8, i < NCH = ceil(H/4), so chunk i of
 * lane l lies in head 4i + l/16 and a head's 128 columns are the 16 lanes of one DPP row: a per-head sum is four DPP
 * steps and a whole-row sum two permlane swaps more. w stays in LDS for the whole workgroup (fp32, zero-padded to
 * NCH*512 columns, in two planes holding columns 0-3 and 4-7 of every chunk, so a lane's 16-byte reads at 16-byte
 * stride are conflict-free). Every row access goes through a buffer descriptor of the row's exact size: the columns
 * past C of the last chunk read 0 and their stores are dropped, and a token outside the table (nc_ve_* entry points)
 * reads a zero-size descriptor, so it mixes in nothing and receives no gradient.
 */
#include "nc_device.h"
#include "nc_internal.h"
#include "nanochat_amd.h"

#include <climits>

namespace nc {
namespace {

constexpr int VE_MAX_HEADS = 16;
constexpr int VE_THREADS = 512;
constexpr int VE_WAVES = VE_THREADS / WAVE;
constexpr int REF_HEADS = 6;   /* the reference kernel's compile-time H (C = 768, ve_gate.cu:34) */

typedef __amdgpu_buffer_rsrc_t Rsrc;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <int H>
struct VeShape {
    static constexpr int C = H * HEAD_DIM;
    static constexpr int NCH = (H + 3) / 4;        /* 8-column chunks per lane */
    static constexpr int Q = NCH * WAVE;           /* chunks per padded row */
    static constexpr int PLANE = H * Q * 4;        /* floats in one LDS plane */
};

/* A descriptor over [p, p + bytes): the wave-uniform operands are taken from the first lane so it lives in SGPRs. */
__device__ __forceinline__ Rsrc row_rsrc(const void *p, int bytes) {
    const unsigned long long u = (unsigned long long)p;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)u), hi = __builtin_amdgcn_readfirstlane((unsigned)(u >> 32));
    return __builtin_amdgcn_make_buffer_rsrc((void *)(((unsigned long long)hi << 32) | lo), (short)0,
                                             __builtin_amdgcn_readfirstlane(bytes), 0x00020000);
}

__device__ __forceinline__ long long uniform64(long long v) {
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)((unsigned long long)v >> 32));
    return (long long)(((unsigned long long)hi << 32) | lo);
}

__device__ __forceinline__ uint4 ld16(Rsrc r, int off) {
    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
    return uint4{v[0], v[1], v[2], v[3]};
}
/* non-temporal: rows streamed once */
__device__ __forceinline__ uint4 ld16_nt(Rsrc r, int off) {
    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 2);
    return uint4{v[0], v[1], v[2], v[3]};
}
__device__ __forceinline__ void st16(Rsrc r, int off, uint4 v) {
    __builtin_amdgcn_raw_buffer_store_b128(u32x4{v.x, v.y, v.z, v.w}, r, off, 0, 0);
}

__device__ __forceinline__ void unpack_bf16x8(uint4 u, float (&x)[8]) {
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int k = 0; k < 4; k++) {
        x[2 * k] = __uint_as_float(w[k] << 16);
        x[2 * k + 1] = __uint_as_float(w[k] & 0xFFFF0000u);
    }
}

__device__ __forceinline__ uint4 pack_bf16x8(const float (&x)[8]) {
    uint32_t w[4];
#pragma unroll
    for (int k = 0; k < 4; k++) w[k] = (uint32_t)f32_to_bf16(x[2 * k]) | ((uint32_t)f32_to_bf16(x[2 * k + 1]) << 16);
    return uint4{w[0], w[1], w[2], w[3]};
}

/* fp32 rounded to bf16 and back (round to nearest even). */
__device__ __forceinline__ float bf16r(float x) { return bf16_to_f32(f32_to_bf16(x)); }

/* Eight fp32 table values (two 16-byte words) rounded to bf16, packed. */
__device__ __forceinline__ uint4 table_bf16x8(uint4 a, uint4 b) {
    const float x[8] = {__uint_as_float(a.x), __uint_as_float(a.y), __uint_as_float(a.z), __uint_as_float(a.w),
                        __uint_as_float(b.x), __uint_as_float(b.y), __uint_as_float(b.z), __uint_as_float(b.w)};
    return pack_bf16x8(x);
}

template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}

/* Sum over each 16-lane row (quad_perm [1,0,3,2], quad_perm [2,3,0,1], row_half_mirror, row_mirror): every lane of
 * the row ends with the same bits, since each step adds the same two partial sums in either order. */
__device__ __forceinline__ float row16_sum(float v) {
    v = v + dpp<0xB1>(v);
    v = v + dpp<0x4E>(v);
    v = v + dpp<0x141>(v);
    v = v + dpp<0x140>(v);
    return v;
}

__device__ __forceinline__ float wave_sum(float v) { return pair_sum32(pair_sum16(row16_sum(v))); }

/* w [H][C] fp32 -> LDS planes: column c of head h, chunk q = c / 8, at plane (c % 8) / 4, float (h Q + q) 4 + c % 4;
 * columns C .. Q*8 are zero. */
template <int H>
__device__ __forceinline__ void stage_w(float *ws, const float *w) {
    using S = VeShape<H>;
    for (int i = threadIdx.x; i < H * S::Q * 2; i += VE_THREADS) {
        const int h = i / (2 * S::Q), q = (i >> 1) % S::Q, half = i & 1, c = q * 8 + half * 4;
        float4 x = {0.0f, 0.0f, 0.0f, 0.0f};
        if (c < S::C) x = *reinterpret_cast<const float4 *>(w + (long long)h * S::C + c);
        *reinterpret_cast<float4 *>(ws + half * S::PLANE + (h * S::Q + q) * 4) = x;
    }
}

template <int H>
__device__ __forceinline__ void w_chunk(const float *ws, int h, int q, float (&wv)[8]) {
    using S = VeShape<H>;
    const float4 a = *reinterpret_cast<const float4 *>(ws + (h * S::Q + q) * 4);
    const float4 b = *reinterpret_cast<const float4 *>(ws + S::PLANE + (h * S::Q + q) * 4);
    wv[0] = a.x; wv[1] = a.y; wv[2] = a.z; wv[3] = a.w;
    wv[4] = b.x; wv[5] = b.y; wv[6] = b.z; wv[7] = b.w;
}

struct VeFwd {
    const uint16_t *n, *v;          /* n: [rows][C]; v: rows at v_stride elements */
    long long v_stride;
    const int32_t *idx;             /* [rows] tokens */
    const float *table;             /* [vocab][C] */
    long long vocab;
    const float *w;                 /* [H][C] */
    uint16_t *out;                  /* [rows][C] */
    float *gate;                    /* [rows][H] */
    long long rows;
};

template <int H>
__global__ void __launch_bounds__(VE_THREADS) ve_forward_kernel(VeFwd a) {
    using S = VeShape<H>;
    constexpr int C = S::C, NCH = S::NCH;
    __shared__ __attribute__((aligned(16))) float ws[2 * S::PLANE];
    stage_w<H>(ws, a.w);
    __syncthreads();
    const int lane = threadIdx.x & (WAVE - 1);
    const long long step = (long long)gridDim.x * VE_WAVES;
    for (long long rr = (long long)blockIdx.x * VE_WAVES + (threadIdx.x >> 6); rr < a.rows; rr += step) {
        const long long r = uniform64(rr);
        const int tok = __builtin_amdgcn_readfirstlane(a.idx[r]);
        const bool ok = tok >= 0 && (long long)tok < a.vocab;
        const Rsrc rn = row_rsrc(a.n + r * C, C * 2), rv = row_rsrc(a.v + r * a.v_stride, C * 2);
        const Rsrc re = row_rsrc(a.table + (ok ? (long long)tok * C : 0), ok ? C * 4 : 0);
        uint4 xn[NCH], xv[NCH], e0[NCH], e1[NCH];
#pragma unroll
        for (int i = 0; i < NCH; i++) {
            const int off = (i * WAVE + lane) * 16;
            xn[i] = ld16_nt(rn, off);
            xv[i] = ld16_nt(rv, off);
            e0[i] = ld16(re, 2 * off);
            e1[i] = ld16(re, 2 * off + 16);
        }
        float x[NCH][8];
#pragma unroll
        for (int i = 0; i < NCH; i++) unpack_bf16x8(xn[i], x[i]);
        /* one head at a time (a loop, not unrolled, so w's LDS reads are not all hoisted into registers); lane h
         * keeps gate h */
        float mine = 0.0f;
#pragma unroll 1
        for (int h = 0; h < H; h++) {
            float z = 0.0f;
#pragma unroll
            for (int i = 0; i < NCH; i++) {
                float wv[8];
                w_chunk<H>(ws, h, i * WAVE + lane, wv);
#pragma unroll
                for (int j = 0; j < 8; j++) z = __builtin_fmaf(x[i][j], wv[j], z);
            }
            const float g = 2.0f * (1.0f / (1.0f + expf(-wave_sum(z))));
            if (lane == h) mine = g;
        }
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(mine), row_rsrc(a.gate + r * H, H * 4), lane * 4, 0, 0);
        const Rsrc ro = row_rsrc(a.out + r * C, C * 2);
#pragma unroll
        for (int i = 0; i < NCH; i++) {
            /* chunk i's head 4i + lane/16 (a lane past the last head reads a gate it multiplies by zeros) */
            const float gh = __shfl(mine, min(4 * i + (lane >> 4), H - 1), WAVE);
            float x[8], e[8];
            unpack_bf16x8(xv[i], x);
            unpack_bf16x8(table_bf16x8(e0[i], e1[i]), e);
#pragma unroll
            for (int j = 0; j < 8; j++) x[j] = x[j] + gh * e[j];
            st16(ro, (i * WAVE + lane) * 16, pack_bf16x8(x));
        }
    }
}

struct VeBwd {
    const uint16_t *dout;           /* rows at dout_stride elements */
    long long dout_stride;
    const int32_t *ids;             /* [rows] tokens in visiting (sorted) order */
    const long long *order;         /* [rows] the row of each position */
    const float *table;             /* [vocab][C] */
    long long vocab;
    const float *w;                 /* [H][C] */
    const float *gate;              /* [rows][H] */
    uint16_t *dn;                   /* [rows][C] */
    float *dtable;                  /* [vocab][C], added into */
    uint16_t *dz;                   /* [rows][H] */
    long long rows;
};

/* w [H][C] fp32 -> LDS unchanged: the backward reads columns (2 lane, 2 lane + 1) of a head, 8 bytes at 8-byte
 * stride, conflict-free. */
template <int H>
__device__ __forceinline__ void stage_w_rows(float *ws, const float *w) {
    for (int i = threadIdx.x; i < H * H * HEAD_DIM / 4; i += VE_THREADS)
        reinterpret_cast<float4 *>(ws)[i] = reinterpret_cast<const float4 *>(w)[i];
}

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

/* The row of dtable is read when a run begins rather than when it ends where registers for it cost no waves: beside a
 * second position's rows (AHEAD, below), and from 13 heads, whose w leaves room for one workgroup a CU in LDS. */
template <int H, bool AHEAD>
constexpr bool VE_EARLY = AHEAD || H * H * HEAD_DIM * 4 > 80 * 1024;

/* The run a wave is in. */
template <int H>
struct VeRun {
    bool started, ok, shared;   /* a run; a token of the table; it began in the wave before */
    int t;
    uint32_t eb[H];             /* the token's table columns as bf16x2 */
    float acc[H][2];
    u32x2 old[H];               /* VE_EARLY: the token's row of dtable before the run */
};

/* A run's accumulated table gradient added into dtable row t. With equal tokens adjacent in `ids` (sorted, the
 * reference's contract), a run that neither starts at the wave's first position nor ends at its last one holds every
 * occurrence of its token, so no other wave touches that row: a plain read-add-write. So does a wave's first or last run
 * when the id before or after its range is another token; otherwise (shared) the run continues in a neighbouring wave's
 * range: hardware fp32 atomics (two instructions per head, each 64 dwords at 8-byte stride). */
template <int H, bool AHEAD>
__device__ __forceinline__ void flush_run(const VeBwd &a, VeRun<H> &run, int lane, bool shared) {
    if (!run.started || !run.ok) return;
    float *row = a.dtable + (long long)run.t * (H * HEAD_DIM) + 2 * lane;
    if (shared) {
#pragma unroll
        for (int k = 0; k < H; k++) {
            unsafeAtomicAdd(row + k * HEAD_DIM, run.acc[k][0]);
            unsafeAtomicAdd(row + k * HEAD_DIM + 1, run.acc[k][1]);
        }
        return;
    }
    if (!VE_EARLY<H, AHEAD>) {
#pragma unroll
        for (int k = 0; k < H; k++) run.old[k] = *reinterpret_cast<const u32x2 *>(row + k * HEAD_DIM);
    }
#pragma unroll
    for (int k = 0; k < H; k++)
        *reinterpret_cast<float2 *>(row + k * HEAD_DIM) =
            float2{__uint_as_float(run.old[k][0]) + run.acc[k][0], __uint_as_float(run.old[k][1]) + run.acc[k][1]};
}

/* Up to 64 positions' rows and tokens, lane l position l's. */
struct VePositions {
    uint32_t row_lo, row_hi;
    int id, n;
};

/* A position's row and token and what it reads of them. e, old: the table's and dtable's row where a run begins. */
template <int H>
struct VeRow {
    long long r;
    int t;
    bool valid, fresh, ok;   /* a row; the first of a run; a token of the table */
    bool shared;             /* fresh: the run began in the wave before */
    uint32_t d[H];
    float g[H];              /* the row's gates; AHEAD: g[0] lane h's of head h */
    u32x2 e[H], old[H];
};

/* The rows of w's token where a run begins (there): the table's and, with OLD, dtable's unless another wave adds to it. */
template <int H, bool OLD>
__device__ __forceinline__ void ve_fetch_run(const VeBwd &a, VeRow<H> &w, bool there, int lane) {
    constexpr int C = H * HEAD_DIM;
    const bool row = there && w.ok;
    const Rsrc re = row_rsrc(a.table + (row ? (long long)w.t * C : 0), row ? C * 4 : 0);
    const Rsrc ro = row_rsrc(a.dtable + (row ? (long long)w.t * C : 0), row && !w.shared ? C * 4 : 0);
#pragma unroll
    for (int k = 0; k < H; k++) {
        w.e[k] = __builtin_amdgcn_raw_buffer_load_b64(re, (k * HEAD_DIM + 2 * lane) * 4, 0, 0);
        if (OLD) w.old[k] = __builtin_amdgcn_raw_buffer_load_b64(ro, (k * HEAD_DIM + 2 * lane) * 4, 0, 0);
    }
}

/* Position q's row, with `run` the token of the run before it (started: there is one). AHEAD: also its gate and, where it
 * begins a run, the token's rows. Loads a position does not need go through zero-size descriptors: no access, and no branch
 * that would make the compiler wait for those in flight. */
template <int H, bool AHEAD>
__device__ __forceinline__ void ve_fetch(const VeBwd &a, const VePositions &ps, int q, bool has_before, int before,
                                         bool started, int run, int lane, VeRow<H> &w) {
    constexpr int C = H * HEAD_DIM;
    const int l = q & (WAVE - 1);
    const uint32_t lo = __builtin_amdgcn_readlane(ps.row_lo, l), hi = __builtin_amdgcn_readlane(ps.row_hi, l);
    w.r = q < ps.n ? (long long)(((unsigned long long)hi << 32) | lo) : -1;
    w.t = __builtin_amdgcn_readlane(ps.id, l);
    w.valid = w.r >= 0 && w.r < a.rows;   /* not a row: nothing to read or write */
    w.fresh = w.valid && (!started || w.t != run);
    w.ok = w.t >= 0 && (long long)w.t < a.vocab;
    w.shared = !started && has_before && w.t == before;
    const Rsrc rd = row_rsrc(a.dout + (w.valid ? w.r * a.dout_stride : 0), w.valid ? C * 2 : 0);
    const float *gate = a.gate + (w.valid ? w.r * H : 0);
    if (AHEAD)
        w.g[0] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(row_rsrc(gate, w.valid ? H * 4 : 0), lane * 4, 0, 0));
#pragma unroll
    for (int k = 0; k < H; k++) {
        w.d[k] = __builtin_amdgcn_raw_buffer_load_b32(rd, (k * HEAD_DIM + 2 * lane) * 2, 0, 2);
        if (!AHEAD) w.g[k] = gate[k];
    }
    if (AHEAD) ve_fetch_run<H, true>(a, w, w.fresh, lane);
}

template <int H, bool AHEAD>
__device__ __forceinline__ void ve_row(const VeBwd &a, const float *ws, VeRow<H> &w, VeRun<H> &run, int lane) {
    constexpr int C = H * HEAD_DIM;
    if (!w.valid) return;
    if (w.fresh) {
        if (!AHEAD) ve_fetch_run<H, VE_EARLY<H, false>>(a, w, true, lane);
        flush_run<H, AHEAD>(a, run, lane, run.shared);
        run.started = true;
        run.shared = w.shared;
        run.t = w.t;
        run.ok = w.ok;
#pragma unroll
        for (int k = 0; k < H; k++) {
            run.eb[k] = (uint32_t)f32_to_bf16(__uint_as_float(w.e[k][0])) |
                        ((uint32_t)f32_to_bf16(__uint_as_float(w.e[k][1])) << 16);
            if (VE_EARLY<H, AHEAD>) run.old[k] = w.old[k];
            run.acc[k][0] = 0.0f;
            run.acc[k][1] = 0.0f;
        }
    }
    float dz[H], mine = 0.0f;
#pragma unroll
    for (int k = 0; k < H; k++) {
        const float g = AHEAD ? __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(w.g[0]), k)) : w.g[k];
        const float d0 = __uint_as_float(w.d[k] << 16), d1 = __uint_as_float(w.d[k] & 0xFFFF0000u);
        const float e0 = __uint_as_float(run.eb[k] << 16), e1 = __uint_as_float(run.eb[k] & 0xFFFF0000u);
        run.acc[k][0] = run.acc[k][0] + bf16r(g * d0);
        run.acc[k][1] = run.acc[k][1] + bf16r(g * d1);
        const float dg = wave_sum(__builtin_fmaf(d1, e1, d0 * e0)), sg = g * 0.5f;
        dz[k] = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(2.0f * dg * (1.0f - sg) * sg)));
        if (lane == k) mine = dz[k];
    }
    __builtin_amdgcn_raw_buffer_store_b16(f32_to_bf16(mine), row_rsrc(a.dz + w.r * H, H * 2), lane * 2, 0, 0);
    const Rsrc rn = row_rsrc(a.dn + w.r * C, C * 2);
    /* dn one head's columns at a time (a loop, so w's LDS reads are not all hoisted into registers) */
#pragma unroll 1
    for (int k = 0; k < H; k++) {
        float x0 = 0.0f, x1 = 0.0f;
#pragma unroll
        for (int h = 0; h < H; h++) {
            const float2 wv = *reinterpret_cast<const float2 *>(ws + h * C + k * HEAD_DIM + 2 * lane);
            x0 = __builtin_fmaf(dz[h], wv.x, x0);
            x1 = __builtin_fmaf(dz[h], wv.y, x1);
        }
        __builtin_amdgcn_raw_buffer_store_b32((uint32_t)f32_to_bf16(x0) | ((uint32_t)f32_to_bf16(x1) << 16), rn,
                                              (k * HEAD_DIM + 2 * lane) * 2, 0, 0);
    }
}

/* Backward mapping (unlike the forward's): lane l holds columns k*128 + 2l and k*128 + 2l + 1 of every head k, so a
 * head's gate is one scalar, dg is a whole-wave sum, and every access of dout, the table, dn and dtable is 4 or 8
 * contiguous bytes per lane, 256 or 512 contiguous bytes per instruction. A position is a chain of loads (its row's
 * number, then the row, then at a run's end the row of dtable: 2.4 us a position), so 64 positions' numbers and tokens
 * are read at once, one a lane. The rest of the chain is hidden by the resident waves or, AHEAD, by loading a position's
 * rows before the arithmetic of the one before it, into a second register set (the loop alternates two by name): 135
 * registers at H = 6 against 72, so fewer waves (choose_backward says where which is the faster). H = 6, tokens of a
 * log-uniform vocabulary, us against one position at a time with every border run atomic: 256 rows 5.5 -> 5.1, 4,096
 * 32 -> 15.5, 16,384 81 -> 34, 65,536 103 -> 88 (its bytes take 84); H = 13 4,096 rows 47 -> 35, 65,536 234 -> 225; H = 16
 * 57 -> 41 and 288 -> 287. */
template <int H, bool AHEAD>
__global__ void __launch_bounds__(VE_THREADS) ve_backward_kernel(VeBwd a) {
    constexpr int C = H * HEAD_DIM;
    __shared__ __attribute__((aligned(16))) float ws[H * C];
    const int lane = threadIdx.x & (WAVE - 1);
    const long long nw = (long long)gridDim.x * VE_WAVES;
    const long long wid = uniform64((long long)blockIdx.x * VE_WAVES + (threadIdx.x >> 6));
    const long long p0 = a.rows * wid / nw, p1 = a.rows * (wid + 1) / nw;
    const bool has_before = p0 > 0 && p0 < p1, has_after = p1 < a.rows && p0 < p1;
    const int before = has_before ? __builtin_amdgcn_readfirstlane(a.ids[p0 - 1]) : 0;
    const int after = has_after ? __builtin_amdgcn_readfirstlane(a.ids[p1]) : 0;
    const auto positions = [&](long long base) {
        VePositions ps;
        ps.n = (int)(p1 - base < WAVE ? p1 - base : WAVE);
        const unsigned long long row = lane < ps.n ? (unsigned long long)a.order[base + lane] : ~0ull;
        ps.row_lo = (uint32_t)row;
        ps.row_hi = (uint32_t)(row >> 32);
        ps.id = lane < ps.n ? a.ids[base + lane] : -1;
        return ps;
    };
    VePositions ps = positions(p0);   /* in flight while w is staged */
    stage_w_rows<H>(ws, a.w);
    __syncthreads();
    VeRun<H> run;
    run.started = run.ok = run.shared = false;
    run.t = -1;
    for (long long base = p0; base < p1; base += WAVE) {
        if (base > p0) ps = positions(base);
        VeRow<H> x, y;
        if (!AHEAD) {
            for (int q = 0; q < ps.n; q++) {
                ve_fetch<H, false>(a, ps, q, has_before, before, run.started, run.t, lane, x);
                ve_row<H, false>(a, ws, x, run, lane);
            }
            continue;
        }
        ve_fetch<H, true>(a, ps, 0, has_before, before, run.started, run.t, lane, x);
        for (int q = 0; q < ps.n; q += 2) {
            ve_fetch<H, true>(a, ps, q + 1, has_before, before, run.started || x.valid, x.valid ? x.t : run.t, lane, y);
            ve_row<H, true>(a, ws, x, run, lane);
            if (q + 1 >= ps.n) break;
            ve_fetch<H, true>(a, ps, q + 2, has_before, before, run.started || y.valid, y.valid ? y.t : run.t, lane, x);
            ve_row<H, true>(a, ws, y, run, lane);
        }
    }
    flush_run<H, AHEAD>(a, run, lane, run.shared || (has_after && run.t == after));
}

/* The gate weight's gradient dw[h][c] = sum over rows of dz[row][h] n[row][c] (bf16 operands, fp32 sums): H <= 16
 * outputs a column, so it is bound by reading n once, not by the products, and a matrix product's tiles (H of 16 rows
 * used, a few column tiles for the whole sum over the rows) leave the chip idle. A block takes a slab of rows and 256
 * columns, a lane four columns of all H heads; 64 rows at a time, 16 a wave, dz through LDS. The waves' and then the
 * slabs' sums are added in a fixed order. 65,536 rows, H = 6: 143 -> 40 us (2.5 TB/s of n) */
struct VeWeight {
    const uint16_t *dz;   /* [rows][H] bf16 */
    const uint16_t *n;    /* [rows][C] bf16 */
    long long rows, per;  /* rows of a slab: a multiple of VW_ROWS */
    float *part;          /* [slabs][H][C] */
};

constexpr int VW_ROWS = 64, VW_COLS = 256, VW_WAVES = 4;
constexpr int VW_PER = VW_ROWS / VW_WAVES;

template <int H>
__global__ void __launch_bounds__(VW_WAVES *WAVE) ve_weight_kernel(VeWeight a) {
    constexpr int C = H * HEAD_DIM;
    __shared__ float z[VW_ROWS * H];
    __shared__ __align__(16) float red[VW_WAVES][VW_COLS];
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x >> 6;
    const int col = blockIdx.y * VW_COLS + lane * 4;
    const bool in = col < C;
    const long long r0 = blockIdx.x * a.per, r1 = r0 + a.per < a.rows ? r0 + a.per : a.rows;
    float acc[H][4];
#pragma unroll
    for (int h = 0; h < H; h++)
#pragma unroll
        for (int e = 0; e < 4; e++) acc[h][e] = 0.0f;
    for (long long r = r0; r < r1; r += VW_ROWS) {
        const int live = (int)(r1 - r < VW_ROWS ? r1 - r : VW_ROWS);
        uint2 x[VW_PER];
#pragma unroll
        for (int k = 0; k < VW_PER; k++) {
            const int row = wave * VW_PER + k;
            x[k] = in && row < live ? *reinterpret_cast<const uint2 *>(a.n + (r + row) * C + col) : uint2{0u, 0u};
        }
        __syncthreads();   /* the rows before are done with z */
        for (int i = threadIdx.x; i < VW_ROWS * H; i += VW_WAVES * WAVE) z[i] = i < live * H ? bf16_to_f32(a.dz[r * H + i]) : 0.0f;
        __syncthreads();
#pragma unroll
        for (int k = 0; k < VW_PER; k++) {
            const float f[4] = {__uint_as_float(x[k].x << 16), __uint_as_float(x[k].x & 0xFFFF0000u),
                                __uint_as_float(x[k].y << 16), __uint_as_float(x[k].y & 0xFFFF0000u)};
#pragma unroll
            for (int h = 0; h < H; h++) {
                const float d = z[(wave * VW_PER + k) * H + h];
#pragma unroll
                for (int e = 0; e < 4; e++) acc[h][e] = __builtin_fmaf(d, f[e], acc[h][e]);
            }
        }
    }
#pragma unroll 1
    for (int h = 0; h < H; h++) {
        float4 v = float4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < H; k++)   /* acc[h] without indexing registers */
            if (k == h) v = float4{acc[k][0], acc[k][1], acc[k][2], acc[k][3]};
        __syncthreads();
        *reinterpret_cast<float4 *>(&red[wave][lane * 4]) = v;
        __syncthreads();
        const int c = blockIdx.y * VW_COLS + threadIdx.x;
        if (c < C)
            a.part[((long long)blockIdx.x * H + h) * C + c] =
                ((red[0][threadIdx.x] + red[1][threadIdx.x]) + red[2][threadIdx.x]) + red[3][threadIdx.x];
    }
}

/* dw from the slabs' partials: 64 outputs a block, group g of 16 adds the g-th sixteenth of the slabs, then the groups in
 * order. */
__global__ void __launch_bounds__(1024) ve_weight_sum_kernel(const float *part, int slabs, int n, float *dw) {
    __shared__ float sums[16][64];
    const int o = threadIdx.x & 63, g = threadIdx.x >> 6, i = blockIdx.x * 64 + o;   /* n is a multiple of 64 */
    const int s0 = slabs * g / 16, s1 = slabs * (g + 1) / 16;
    float sum = 0.0f;
#pragma unroll 8
    for (int s = s0; s < s1; s++) sum = sum + part[(long long)s * n + i];
    sums[g][o] = sum;
    __syncthreads();
    if (g) return;
    for (int k = 1; k < 16; k++) sum = sum + sums[k][o];
    dw[i] = sum;
}

/* Slabs of `rows` rows for H heads, none of fewer than VW_ROWS rows: as many as run at once, four workgroups a CU, or three
 * from 11 heads, whose 132 registers and more leave room for no fourth (with four, 16,384 rows of 13 heads ran a second round
 * of 128 of their 896 workgroups: 36 us, now 31; 65,536 98 -> 75). */
void ve_weight_slabs(long long rows, int heads, int &slabs, long long &per) {
    const int chunks = (heads * HEAD_DIM + VW_COLS - 1) / VW_COLS;
    const long long tiles = (rows + VW_ROWS - 1) / VW_ROWS, most = (heads <= 10 ? 1024 : 768) / chunks;
    const long long want = tiles < most ? tiles : most;
    per = (tiles + want - 1) / want * VW_ROWS;
    slabs = (int)((rows + per - 1) / per);
}

template <int H = 1>
int launch_weight(int heads, const VeWeight &a, int slabs, float *dw, hipStream_t stream) {
    if constexpr (H > VE_MAX_HEADS) {
        return NC_ERR_SHAPE;
    } else {
        if (heads != H) return launch_weight<H + 1>(heads, a, slabs, dw, stream);
        constexpr int C = H * HEAD_DIM;
        hipLaunchKernelGGL(ve_weight_kernel<H>, dim3(slabs, (C + VW_COLS - 1) / VW_COLS), dim3(VW_WAVES * WAVE), 0,
                           stream, a);
        hipLaunchKernelGGL(ve_weight_sum_kernel, dim3(H * C / 64), dim3(1024), 0, stream, a.part, slabs, H * C, dw);
        return (int)hipGetLastError();
    }
}

constexpr int VE_MOST = 8;   /* workgroups of VE_THREADS that a CU holds, and more */

/* Workgroups for `rows` rows: `per` rows a wave, at most as many workgroups as the device holds at once, `most` a CU (the
 * kernel's resident workgroups per device, cached per device in `resident`). */
template <typename K>
int ve_blocks(K kernel, long long rows, int per, int most, int (&resident)[64]) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return -1;
    if (!resident[dev]) {
        int cus = 0, per_cu = 0;
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, VE_THREADS, 0) != hipSuccess)
            return -1;
        resident[dev] = max(1, cus) * max(1, min(per_cu, most));
    }
    const long long need = (rows + VE_WAVES * per - 1) / (VE_WAVES * per);
    return (int)max(1LL, min(need, (long long)resident[dev]));
}

template <int H>
int launch_forward(const VeFwd &a, hipStream_t stream) {
    static int resident[64] = {0};
    const int blocks = ve_blocks(ve_forward_kernel<H>, a.rows, 1, VE_MOST, resident);
    if (blocks < 0) return (int)hipErrorInvalidDevice;
    hipLaunchKernelGGL(ve_forward_kernel<H>, dim3(blocks), dim3(VE_THREADS), 0, stream, a);
    return (int)hipGetLastError();
}

template <int H, bool AHEAD>
int launch_backward(const VeBwd &a, int per, hipStream_t stream) {
    static int resident[64] = {0};
    const int blocks = ve_blocks(ve_backward_kernel<H, AHEAD>, a.rows, per, AHEAD ? 3 : VE_MOST, resident);
    if (blocks < 0) return (int)hipErrorInvalidDevice;
    hipLaunchKernelGGL((ve_backward_kernel<H, AHEAD>), dim3(blocks), dim3(VE_THREADS), 0, stream, a);
    return (int)hipGetLastError();
}

constexpr int VE_AHEAD_HEADS = 10;

/* The form, and rows a wave, at most four while every wave finds that many.
 * Rows a wave: a frequent token's rows all add into one row of dtable, a wave at a time, so more waves mean more adds at the
 * same addresses; fewer leave the chip idle (H = 6, one / two / four rows a wave: 1,024 rows 8.8 / 7.7 / 10.9 us, 4,096
 * 26 / 17 / 15).
 * The second register set wins where a wave has several rows but the waves do not fill the chip, and at few heads always
 * (AHEAD / not, us of log-uniform tokens, caches cold: H = 6 1,024 rows 14.9 / 13.8, 2,048 17.2 / 18.4, 4,096 22.2 / 24.6,
 * 32,768 68 / 78, 65,536 119 / 108; H = 2 4,096 14.0 / 15.3, 65,536 53 / 61; H = 5, warm, 65,536 76 / 87; H = 8 4,096
 * 27.3 / 29.4, 32,768 84 / 83, 65,536 145 / 131; H = 10 4,096 33.8 / 34.3, 16,384 66 / 72, 32,768 107 / 102, 65,536 182 /
 * 156). From 11 heads it takes 253 registers, from 13 it spilled: 65,536 rows of 16 heads took 931 us. At one and two heads
 * it fits a fourth workgroup a CU, whose adds cost more than it brings (65,536 rows, H = 1: 46 us with four, 36 with three). */
template <int H>
int choose_backward(const VeBwd &a, hipStream_t stream) {
    const int per = (int)max(1LL, min(4LL, a.rows / 1024));
    if constexpr (H <= VE_AHEAD_HEADS) {
        const long long end = H <= 5 ? LLONG_MAX : H <= 8 ? 49152 : 24576;
        if (a.rows >= (H <= 2 ? 0 : 2048) && a.rows < end) return launch_backward<H, true>(a, per, stream);
    }
    return launch_backward<H, false>(a, per, stream);
}

template <int H = 1>
int dispatch(int heads, bool fwd, const VeFwd &f, const VeBwd &b, hipStream_t stream) {
    if constexpr (H > VE_MAX_HEADS) {
        return NC_ERR_SHAPE;
    } else {
        if (heads == H) return fwd ? launch_forward<H>(f, stream) : choose_backward<H>(b, stream);
        return dispatch<H + 1>(heads, fwd, f, b, stream);
    }
}

bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

int check_forward(const VeFwd &a, int heads) {
    if (heads < 1 || heads > VE_MAX_HEADS || a.rows < 0 || a.vocab < 1 || a.v_stride < (long long)heads * HEAD_DIM ||
        a.v_stride % 8)
        return NC_ERR_SHAPE;
    if (a.rows == 0) return NC_OK;
    if (!a.n || !a.v || !a.idx || !a.table || !a.w || !a.out || !a.gate) return NC_ERR_NULL;
    if (!aligned16(a.n) || !aligned16(a.v) || !aligned16(a.table) || !aligned16(a.w) || !aligned16(a.out) ||
        ((uintptr_t)a.gate & 3))
        return NC_ERR_SHAPE;
    return NC_OK;
}

int check_backward(const VeBwd &a, int heads) {
    if (heads < 1 || heads > VE_MAX_HEADS || a.rows < 0 || a.vocab < 1 ||
        a.dout_stride < (long long)heads * HEAD_DIM || a.dout_stride % 8)
        return NC_ERR_SHAPE;
    if (a.rows == 0) return NC_OK;
    if (!a.dout || !a.ids || !a.order || !a.table || !a.w || !a.gate || !a.dn || !a.dtable || !a.dz)
        return NC_ERR_NULL;
    if (!aligned16(a.dout) || !aligned16(a.table) || !aligned16(a.w) || !aligned16(a.dn) || !aligned16(a.dtable) ||
        ((uintptr_t)a.gate & 3) || ((uintptr_t)a.dz & 1) || ((uintptr_t)a.order & 7))
        return NC_ERR_SHAPE;
    return NC_OK;
}

int ve_forward_run(const VeFwd &a, int heads, hipStream_t stream) {
    const int st = check_forward(a, heads);
    if (st != NC_OK || a.rows == 0) return st;
    return dispatch(heads, true, a, VeBwd{}, stream);
}

int ve_backward_run(const VeBwd &a, int heads, hipStream_t stream) {
    const int st = check_backward(a, heads);
    if (st != NC_OK || a.rows == 0) return st;
    return dispatch(heads, false, VeFwd{}, a, stream);
}

VeFwd forward_args(const void *n, const void *v, long long v_stride, const void *idx, const void *table,
                   long long vocab, const void *w, void *out, void *gate, long long rows) {
    return VeFwd{(const uint16_t *)n, (const uint16_t *)v, v_stride, (const int32_t *)idx, (const float *)table, vocab,
                 (const float *)w, (uint16_t *)out, (float *)gate, rows};
}

VeBwd backward_args(const void *dout, long long dout_stride, const void *ids, const void *order, const void *table,
                    long long vocab, const void *w, const void *gate, void *dn, void *dtable, void *dz, long long rows) {
    return VeBwd{(const uint16_t *)dout, dout_stride, (const int32_t *)ids, (const long long *)order,
                 (const float *)table, vocab, (const float *)w, (const float *)gate, (uint16_t *)dn, (float *)dtable,
                 (uint16_t *)dz, rows};
}

}  // namespace
}  // namespace nc

using namespace nc;

/* The table's row count is not an argument of the reference's entry points: tokens are trusted, as there. */
static constexpr long long UNCHECKED_VOCAB = 0x7FFFFFFFLL;

extern "C" void ve_forward(const void *n, const void *v, long long v_stride, const void *idx, const void *table,
                           const void *w, void *out, void *gate, long long rows, void *stream) {
    set_last_error(ve_forward_run(forward_args(n, v, v_stride, idx, table, UNCHECKED_VOCAB, w, out, gate, rows),
                                  REF_HEADS, (hipStream_t)stream));
}

extern "C" void ve_backward(const void *dout, long long dout_stride, const void *ids, const void *order,
                            const void *table, const void *w, const void *gate, void *dn, void *dtable, void *dz,
                            long long rows, void *stream) {
    set_last_error(ve_backward_run(backward_args(dout, dout_stride, ids, order, table, UNCHECKED_VOCAB, w, gate, dn,
                                                 dtable, dz, rows),
                                   REF_HEADS, (hipStream_t)stream));
}

extern "C" int nc_ve_forward(const void *n, const void *v, long long v_stride, const int32_t *idx, const float *table,
                             long long vocab, const float *w, void *out, float *gate, long long rows, int heads,
                             void *stream) {
    return ve_forward_run(forward_args(n, v, v_stride, idx, table, vocab, w, out, gate, rows), heads,
                          (hipStream_t)stream);
}

extern "C" int nc_ve_backward(const void *dout, long long dout_stride, const int32_t *ids, const int64_t *order,
                              const float *table, long long vocab, const float *w, const float *gate, void *dn,
                              float *dtable, void *dz, long long rows, int heads, void *stream) {
    return ve_backward_run(backward_args(dout, dout_stride, ids, order, table, vocab, w, gate, dn, dtable, dz, rows),
                           heads, (hipStream_t)stream);
}

extern "C" long long nc_ve_weight_grad_workspace_bytes(long long rows, int heads) {
    if (rows < 0 || rows > (1LL << 40) || heads < 1 || heads > VE_MAX_HEADS) return -1;
    if (rows == 0) return 0;
    int slabs;
    long long per;
    ve_weight_slabs(rows, heads, slabs, per);
    return (long long)slabs * heads * heads * HEAD_DIM * 4;
}

extern "C" int nc_ve_weight_grad(const void *dz, const void *n, long long rows, int heads, float *dw, void *workspace,
                                 long long workspace_bytes, void *stream) {
    const long long need = nc_ve_weight_grad_workspace_bytes(rows, heads);
    if (need <= 0) return NC_ERR_SHAPE;   /* no rows: the caller's zeros */
    if (!dz || !n || !dw || !workspace) return NC_ERR_NULL;
    if (((uintptr_t)n & 7) || ((uintptr_t)dz & 1) || (((uintptr_t)dw | (uintptr_t)workspace) & 3)) return NC_ERR_SHAPE;
    if (workspace_bytes < need) return NC_ERR_WORKSPACE;
    VeWeight a;
    a.dz = (const uint16_t *)dz; a.n = (const uint16_t *)n;
    a.rows = rows;
    int slabs;
    ve_weight_slabs(rows, heads, slabs, a.per);
    a.part = (float *)workspace;
    return launch_weight(heads, a, slabs, dw, (hipStream_t)stream);
}
