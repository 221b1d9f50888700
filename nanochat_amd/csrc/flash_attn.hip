/*
 * Training attention for gfx950: the varlen causal (optionally windowed) attention forward that the reference runs
 * through FlashAttention-4 (model/ops/flash_attn.py:325-347: _flash_attn_fwd over cu_seqlens with causal=True,
 * window_size_left = window, return_lse=True; window semantics fa4_window_left, flash_attn.py:309-311).
 *
 * Per segment s (tokens cu[s] .. cu[s+1]-1) and head h, row i attends keys j with j <= i and i - j <= window
 * (window < 0: no left limit):
 *   out[i] = sum_j softmax_j(scale q_i . k_j) v_j          bf16, fp32 accumulation
 *   lse[h][i] = ln sum_j exp(scale q_i . k_j)              fp32 (FA4's (H, total) layout)
 *
 * Mapping: a workgroup of four waves owns 128 query rows of one (segment, head), each wave 32. Keys
 * are visited in blocks of 64, staged in LDS for the four waves (K and V row-major with 16-byte chunks XOR-swizzled
 * by the key) by LDS DMA straight from HBM, in two LDS stages: block b+1 is fetched into one while block b is read
 * from the other, with no registers held for the fetch. Scores are S^T = K Q^T (v_mfma_f32_32x32x16_bf16, keys as
 * rows, queries as columns), so a lane's scores all belong to one query; the online softmax runs in the log2 domain
 * with the lazy rescale of the decode kernels (the reference max moves only when a column's max passes it by 2^8);
 * P^T then feeds O^T += V^T P^T with no shuffle: the V^T operand is read from the row-major tile by gfx950's
 * transposing LDS read (ds_read_b64_tr_b16) in P's key order. The backward stages its Q, dO (or K, V) tiles the
 * same way and reads their transposes the same way.
 */
#include "nc_device.h"
#include "nanochat_amd.h"

namespace nc {
namespace {

constexpr int FA_BM = 128;          /* query rows per workgroup */
constexpr int FA_BN = 64;           /* keys per block */
constexpr int FA_THREADS = 256;
constexpr float FA_LOG2E = 1.4426950408889634f;
constexpr float FA_LN2 = 0.6931471805599453f;
constexpr float FA_RESCALE = 8.0f;  /* lazy rescale threshold (log2 units) */

typedef __amdgpu_buffer_rsrc_t Rsrc;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct FlashFwd {
    const uint16_t *q, *k, *v;      /* (total, H, 128) at token strides q_stride, k_stride, v_stride (elements) */
    long long q_stride, k_stride, v_stride;
    const int32_t *cu;              /* [segments + 1] */
    int segments, H, window;
    float scale_log2;               /* softmax scale * log2(e) */
    uint16_t *out;                  /* (total, H, 128) contiguous */
    float *lse;                     /* [H][lse_stride] */
    long long lse_stride;
};

struct FaStage {
    uint16_t k[FA_BN * HEAD_DIM];   /* [key][128], 16-byte chunk c of key j at chunk c ^ k_swizzle(j) */
    uint16_t v[FA_BN * HEAD_DIM];   /* the same layout: read transposed by ds_read_b64_tr_b16 */
};

/* A row is 256 bytes, all 64 banks, so where rows meet in one access they need different chunks. A row operand's 16 lanes
 * read one chunk of 16 rows: any one-to-one map of row % 16 does. A transposing read's 32 lanes read the same four chunks
 * of four rows r0 .. r0 + 3 (r0 a multiple of 4), so the row's low two bits pick the group of four chunks. With chunk
 * c ^ (row & 15) those rows met in one group: each such read waited 6 cycles, 53 % of the dK/dV kernel's LDS cycles
 * (none now). */
__device__ __forceinline__ int k_swizzle(int row) { return ((row & 3) << 2) | ((row >> 2) & 3); }
__device__ __forceinline__ int k_lds(int row, int chunk) { return row * HEAD_DIM + ((chunk ^ k_swizzle(row)) << 3); }

__device__ __forceinline__ Rsrc make_rsrc(const void *p, unsigned bytes) {
    const unsigned long long u = (unsigned long long)p;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)u), hi = __builtin_amdgcn_readfirstlane((unsigned)(u >> 32));
    return __builtin_amdgcn_make_buffer_rsrc((void *)(((unsigned long long)hi << 32) | lo), (short)0,
                                             __builtin_amdgcn_readfirstlane(bytes), 0x00020000);
}

__device__ __forceinline__ uint4 bload(Rsrc r, int off) {
    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
    return uint4{v[0], v[1], v[2], v[3]};
}

/* Descriptor over `rows` rows of one head starting at token row0: row i at i * stride elements. */
__device__ __forceinline__ Rsrc rows_rsrc(const uint16_t *base, long long row0, long long stride, int h, int rows) {
    const unsigned bytes = rows > 0 ? (unsigned)(((long long)(rows - 1) * stride + HEAD_DIM) * 2) : 0u;
    return make_rsrc(base + row0 * stride + (long long)h * HEAD_DIM, bytes);
}

typedef __attribute__((address_space(3))) void LdsVoid;
typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4i16 LdsV4;

/* A 64-row tile of one head straight into LDS in the k_lds layout by LDS DMA (no registers held), shared by NW
 * waves: instruction i of a wave writes rows 4 i' .. 4 i' + 3 (i' = wave + NW i), lane l the 16 bytes at LDS chunk
 * l % 16 of row 4 i' + l / 16, fetched from the row's chunk (l % 16) ^ k_swizzle(row). Rows past the descriptor's range
 * read zeros. */
template <int NW = 4>
__device__ __forceinline__ void tile_dma(const uint16_t *base, long long row0, long long stride, int h, int rows,
                                         uint16_t *lds, int wave, int lane) {
    const Rsrc rs = rows_rsrc(base, row0, stride, h, rows);
#pragma unroll
    for (int k = 0; k < FA_BN / 4 / NW; k++) {
        const int i = wave + NW * k, r = 4 * i + (lane >> 4), p = lane & 15;
        const int off = (int)((r * stride + ((p ^ k_swizzle(r)) << 3)) * 2);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (LdsVoid *)(lds + i * 4 * HEAD_DIM), 16, off, 0, 0, 0);
    }
}

typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ f32x16 mfma32x32x16(const bf16x8 &a, const bf16x8 &b, const f32x16 &c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

/* A lane's byte offsets into a row-major (k_lds) tile for the A operands of 32 x 32 products; every operand lies at an
 * offset's xor with a constant, plus a constant, so two registers address them all.
 * rows_at: the products over the dimension; lane (hf, c) = (lane / 32, lane % 32) holds dims 16 cc + 8 hf .. +7 of row
 * 32 rt + c. tr_at: the products over 16 rows r0 .. r0 + 15, in the row order of a score tile's registers: lane (hf, c) gets
 * rows r0 + 4 hf .. + 3, then r0 + 8 + 4 hf .. + 3, of dim 32 dt + c. ds_read_b64_tr_b16 hands lane i of a 16-lane group
 * element i % 4 of the 8 bytes lane 4 t + i / 4 points at, for t = 0..3: so lane i points at row base + i / 4, dims
 * 4 (i % 4) .. + 3 of its group's 16. */
__device__ __forceinline__ uint32_t rows_at(int lane) { return 2 * k_lds(lane & 31, lane >> 5); }

__device__ __forceinline__ uint32_t tr_at(int lane) {
    const int i = lane & 15, row = 4 * (lane >> 5) + (i >> 2), dim = (lane & 16) + 4 * (i & 3);
    return 2 * (k_lds(row, dim >> 3) + (dim & 4));
}

typedef __attribute__((address_space(3))) const unsigned char LdsByte;
typedef __attribute__((address_space(3))) const bf16x8 LdsOp;

__device__ __forceinline__ bf16x8 rows_operand32(const uint16_t *tile, uint32_t at, int rt, int cc) {
    return *(LdsOp *)((LdsByte *)tile + (at ^ (cc << 5)) + rt * 32 * HEAD_DIM * 2);
}

__device__ __forceinline__ bf16x8 tr_operand32(const uint16_t *tile, uint32_t at, int dt, int r0) {
    LdsByte *p = (LdsByte *)tile + r0 * HEAD_DIM * 2;
    const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsV4 *)(p + (at ^ (dt << 6))));
    const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsV4 *)(p + (at ^ (dt << 6) ^ 32) + 8 * HEAD_DIM * 2));
    const uint2 x = __builtin_bit_cast(uint2, lo), y = __builtin_bit_cast(uint2, hi);
    return __builtin_bit_cast(bf16x8, uint4{x.x, x.y, y.x, y.y});
}

__device__ __forceinline__ void store4(uint16_t *p, const f32x4 &v, float mul) {
    *reinterpret_cast<uint2 *>(p) = uint2{(uint32_t)f32_to_bf16(v[0] * mul) | ((uint32_t)f32_to_bf16(v[1] * mul) << 16),
                                          (uint32_t)f32_to_bf16(v[2] * mul) | ((uint32_t)f32_to_bf16(v[3] * mul) << 16)};
}

/* The schedule of N products in source order, each with the READS LDS reads of its row or transposed operand four products
 * ahead (two to four measured the same in the dK/dV kernel, six 3 % slower). Left to itself the compiler read an operand
 * right before its product. */
template <int N, int READS>
__device__ __forceinline__ void products_in_order() {
    __builtin_amdgcn_sched_group_barrier(0x100, 4 * READS, 0);
#pragma unroll
    for (int m = 0; m < N; m++) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (m < N - 4) __builtin_amdgcn_sched_group_barrier(0x100, READS, 0);
    }
}

struct FaState {
    f32x16 o[4];   /* O^T tile d: dims 32 d + 8 j + 4 hf + i of column (lane & 31) in registers 4 j + i */
    float m;       /* the column's reference max (log2 domain), equal in both halves */
    float l;       /* sum of exp2(s - m) over the keys this lane's half holds */
};

/* One key block for the wave's 32 queries. kb0: the block's first key (segment-relative); qi: the lane's query row
 * (segment-relative). MASKED: apply causal, window and segment-end bounds per score.
 * Bound by the matrix cores and the exponentials' issue together, at the clock the power limit leaves. 32 x 32 products
 * read K from LDS once for the wave's 32 queries (two 16-wide tiles read it twice) and a column's maximum needs one
 * exchange, not two; blocks no row of a wave sees are skipped. 2 segments of 8,192 tokens x 6 heads: 280 -> 234 us;
 * 8 x 2,048 x 10 heads, window 512: 80 -> 73; 5 x 3,000 x 4: 89 -> 71; 32 x 2,048 x 6, where HBM traffic takes its share of
 * the power: 346 -> 338. Measured slower: the second tile's products among the first one's maxima, the second half's
 * exponentials among the first half's PV products (+ 3 %), a raised wave priority around the scores (+ 4 %). */
template <bool MASKED>
__device__ __forceinline__ void fa_block(const FlashFwd &a, const FaStage &s, const bf16x8 (&qb)[8], FaState &st,
                                         uint32_t rat, uint32_t tat, int kb0, int qi, int seglen, int hf) {
    f32x16 sc[2];
#pragma unroll
    for (int kt = 0; kt < 2; kt++)
#pragma unroll
        for (int i = 0; i < 16; i++) sc[kt][i] = 0.0f;
#pragma unroll
    for (int kt = 0; kt < 2; kt++)
#pragma unroll
        for (int cc = 0; cc < 8; cc++) sc[kt] = mfma32x32x16(rows_operand32(s.k, rat, kt, cc), qb[cc], sc[kt]);
    products_in_order<16, 1>();   /* tile 0's scores, then tile 1's */
    /* raw scores: the scale is positive, so the max of the scaled scores is the scaled max, and it is folded into
     * one FMA per exponential below */
    if (MASKED) {
#pragma unroll
        for (int kt = 0; kt < 2; kt++)
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int key = kb0 + 32 * kt + 8 * (i >> 2) + 4 * hf + (i & 3);
                const bool ok = (key <= qi) & (key < seglen) & ((a.window < 0) | (qi - key <= a.window));
                sc[kt][i] = ok ? sc[kt][i] : -INFINITY;
            }
    }
    float mt = sc[0][0];
#pragma unroll
    for (int i = 1; i < 32; i++) mt = fmaxf(mt, sc[i >> 4][i & 15]);
    mt = pair_max32(mt) * a.scale_log2;
    const float mnew = fmaxf(st.m, mt);
    if (__any(mnew > st.m + FA_RESCALE)) {
        const float alpha = mnew == st.m ? 1.0f : __builtin_amdgcn_exp2f(st.m - mnew);
#pragma unroll
        for (int d = 0; d < 4; d++) st.o[d] *= alpha;
        st.l *= alpha;
        st.m = mnew;
    }
    const float mbase = st.m == -INFINITY ? 0.0f : st.m;
    bf16x8 pv[4];
    float psum = 0.0f;
#pragma unroll
    for (int i = 0; i < 32; i++) {
        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[i >> 4][i & 15], a.scale_log2, -mbase));
        psum += p;
        pv[i >> 3][i & 7] = (__bf16)p;
    }
    st.l += psum;
    /* k-step s2: the half's keys 16 s2 + 4 hf .. + 3 and 16 s2 + 8 + 4 hf .. + 3 */
#pragma unroll
    for (int s2 = 0; s2 < 4; s2++)
#pragma unroll
        for (int d = 0; d < 4; d++) st.o[d] = mfma32x32x16(tr_operand32(s.v, tat, d, 16 * s2), pv[s2], st.o[d]);
    products_in_order<16, 2>();
}

/* A workgroup's (rank, segment, head) from its place in the launch order: work-groups start in linear order (x,
 * then y, then z), so rank r = L / (segments heads) takes the r-th tile of every (segment, head) before any takes
 * the (r + 1)-th. The kernels map rank 0 to their longest tile, so the short ones of every head come last, where they
 * fill the CUs the long ones leave (the grid keeps x = tiles, y = segments, z = heads). Two workgroups share a CU: an XCD
 * (work-groups L % 8) gives its 32 CUs one each, then a second, so the second 32 are taken in reverse, which puts its
 * shortest beside the longest; every later one goes to the CU that is free first. In order, the first CUs' two tiles alone
 * could pass the mean work of a CU: 1 x 8,192 tokens x 6 heads forward 171 -> 166 us, backward 468 -> 455; 5 x 3,000 x 4
 * 72 -> 69, 200 -> 193; 2 x 8,192 x 6 663 -> 654; six rounds of workgroups (32 x 2,048 x 6) the same. */
constexpr unsigned FA_XCDS = 8, FA_XCD_CUS = 32;

struct FaBlock {
    int rank, seg, h;
};

__device__ __forceinline__ FaBlock fa_block_order() {
    const unsigned pairs = gridDim.y * gridDim.z, all = gridDim.x * pairs;
    unsigned L = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
    const unsigned n = L / FA_XCDS, end = min(2 * FA_XCD_CUS, all / FA_XCDS);   /* the n-th of its XCD; whole rows of 8 */
    if (n >= FA_XCD_CUS && n < end) L = (FA_XCD_CUS + end - 1 - n) * FA_XCDS + L % FA_XCDS;
    const unsigned r = L % pairs;
    return FaBlock{(int)(L / pairs), (int)(r % gridDim.y), (int)(r / gridDim.y)};
}

__global__ void __launch_bounds__(FA_THREADS, 2) flash_fwd_kernel(FlashFwd a) {
    __shared__ FaStage st0, st1;   /* distinct objects: a read of one never waits for DMA into the other */
    const FaBlock fb = fa_block_order();
    const int seg = fb.seg, h = fb.h;
    const long long start = a.cu[seg];
    const int seglen = a.cu[seg + 1] - a.cu[seg];
    const int tile = (int)gridDim.x - 1 - fb.rank;   /* the longest key ranges first */
    const int qa = tile * FA_BM;
    if (seglen <= 0 || qa >= seglen) return;
    const int t = threadIdx.x, lane = t & (WAVE - 1), hf = lane >> 5, c = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);   /* in a scalar register, as are the bounds made of it */
    const int qb = min(qa + FA_BM, seglen) - 1;
    const int q0 = qa + wave * 32;                                 /* the wave's first row */
    const bool active = q0 < seglen;
    const int qw1 = min(q0 + 31, seglen - 1);                       /* the wave's last valid row */

    /* the wave's queries: B operand of S^T = K Q^T, lane (hf, c) holds dims 16 cc + 8 hf .. +7 of row c */
    bf16x8 qb_[8];
    {
        const Rsrc rq = rows_rsrc(a.q, start + q0, a.q_stride, h, active ? min(32, seglen - q0) : 0);
#pragma unroll
        for (int cc = 0; cc < 8; cc++)
            qb_[cc] = __builtin_bit_cast(bf16x8, bload(rq, (int)((c * a.q_stride + cc * 16 + hf * 8) * 2)));
    }
    FaState st;
#pragma unroll
    for (int d = 0; d < 4; d++)
#pragma unroll
        for (int i = 0; i < 16; i++) st.o[d][i] = 0.0f;
    st.m = -INFINITY;
    st.l = 0.0f;

    const int klo = a.window >= 0 ? max(0, qa - a.window) : 0;
    const int kb_lo = klo / FA_BN, kb_hi = qb / FA_BN;
    /* block kb + 1 is fetched by LDS DMA into the other stage while block kb is computed; the barrier after the
     * compute (its fence waits for this wave's DMA) makes the fetched block visible and frees the one just read */
    auto fetch = [&](int kb, FaStage &stg) {
        const int n = min(FA_BN, seglen - kb * FA_BN);
        tile_dma(a.k, start + kb * FA_BN, a.k_stride, h, n, stg.k, wave, lane);
        tile_dma(a.v, start + kb * FA_BN, a.v_stride, h, n, stg.v, wave, lane);
    };
    const uint32_t rat = rows_at(lane), tat = tr_at(lane);
    auto compute = [&](int kb, const FaStage &stg) {
        const int k0 = kb * FA_BN, k1 = k0 + FA_BN - 1;
        if (!active || k0 > qw1 || (a.window >= 0 && q0 - k1 > a.window)) return;   /* no row sees the keys */
        /* unmasked iff every key of the block is visible to every row of the wave */
        const bool interior = k1 <= q0 && k1 < seglen && (a.window < 0 || qw1 - k0 <= a.window);
        if (interior)
            fa_block<false>(a, stg, qb_, st, rat, tat, k0, q0 + c, seglen, hf);
        else
            fa_block<true>(a, stg, qb_, st, rat, tat, k0, q0 + c, seglen, hf);
    };
    fetch(kb_lo, st0);
    __syncthreads();
    for (int kb = kb_lo; kb <= kb_hi; kb += 2) {
        if (kb + 1 <= kb_hi) fetch(kb + 1, st1);
        compute(kb, st0);
        __syncthreads();
        if (kb + 1 > kb_hi) break;
        if (kb + 2 <= kb_hi) fetch(kb + 2, st0);
        compute(kb + 1, st1);
        __syncthreads();
    }
    if (!active) return;

    /* out = O^T / l, lse = (m + log2 l) ln 2 */
    const float l = pair_sum32(st.l);
    if (q0 + c >= seglen) return;
    const long long tok = start + q0 + c;
    const float inv = 1.0f / l;
    uint16_t *o = a.out + (tok * a.H + h) * HEAD_DIM + 4 * hf;
#pragma unroll
    for (int d = 0; d < 4; d++)
#pragma unroll
        for (int j = 0; j < 4; j++)
            store4(o + d * 32 + 8 * j, f32x4{st.o[d][4 * j], st.o[d][4 * j + 1], st.o[d][4 * j + 2], st.o[d][4 * j + 3]}, inv);
    if (hf == 0) a.lse[(long long)h * a.lse_stride + tok] = (st.m + __log2f(l)) * FA_LN2;
}

/* ---------------------------------------------------------------------------------------------------------------
 * Backward (the reference's _flash_attn_bwd / bwd_bf16dq, model/ops/flash_attn.py:367-391), per segment and head:
 *   P = exp(scale S - lse), dV = P^T dO, dP = dO V^T, dS = P (dP - D) with D_i = dO_i . O_i (the caller's row
 *   statistics: the reference's `rows`, from the o_proj backward epilogue), dQ = scale dS K, dK = scale dS^T Q.
 * Two kernels and no atomics: flash_bwd_dkv_kernel owns 128 keys (a wave 32) and walks the query blocks that see them;
 * flash_bwd_dq_kernel owns 128 queries (a wave 32, as the forward) and walks their key blocks. S and dP are computed
 * in both (seven 128-deep products per (query, key) pair instead of five), the price of writing dQ once.
 * ------------------------------------------------------------------------------------------------------------- */

struct FlashBwd {
    const uint16_t *q, *k, *v, *dout;         /* (total, H, 128) at token strides */
    long long q_stride, k_stride, v_stride, do_stride;
    const float *lse;                          /* [H][lse_stride], natural log */
    long long lse_stride;
    const float *dpsum;                        /* (total, H): D = dO . O per row */
    const int32_t *cu;
    int segments, H, window;
    float scale, scale_log2;
    uint16_t *dq, *dk, *dv;                    /* (total, H, 128) at their token strides */
    long long dq_stride, dk_stride, dv_stride;
};

/* bitwise, not short-circuit: evaluated per element inside unrolled loops, a branch per term would split the wave */
__device__ __forceinline__ bool visible(int key, int q, int seglen, int window) {
    return (key <= q) & (q < seglen) & ((window < 0) | (q - key <= window));
}

struct alignas(16) DkvStage {
    uint16_t q[FA_BN * HEAD_DIM], dout[FA_BN * HEAD_DIM];   /* k_lds layout; Q^T and dO^T read transposed */
    float nlse[FA_BN], nd[FA_BN];              /* the block's rows: -lse / scale (-inf past the segment), -D */
};

/* dK, dV of 128 keys, 32 a wave: S = Q K^T and dP = dO V^T in 32 x 32 tiles with queries as rows (a lane holds one key's
 * column), so P and dS feed dV^T += dO^T P and dK^T += Q^T dS directly as B operands, with dO^T and Q^T read transposed from
 * the staged tiles. A wave's 32 columns make every operand read from LDS feed twice the products that 16 x 16 tiles of 16
 * keys a wave did: those read 64 KiB a wave and block for 64 products, twice the time of the products themselves.
 * Two blocks of four waves share a CU. At 65,536 tokens of 2,048-token segments x 6 heads dK/dV went from 675 us by trace (16 x
 * 16 tiles in blocks of eight waves) to 546, and with k_swizzle to 464; the backward with these tiles alone 912 -> 810, at
 * 2 x 8,192 tokens 762 -> 690, at 8 x 2,048 x 10 heads with a window of 512 232 -> 208. */
constexpr int DKV_WAVES = 4;
constexpr int DKV_KEYS = 32 * DKV_WAVES;
constexpr int DKV_PARKED = 3;   /* K's last operand and V's last two wait in LDS: 256 registers hold the other 13 */

__global__ void __launch_bounds__(64 * DKV_WAVES, 2) flash_bwd_dkv_kernel(FlashBwd a) {
    __shared__ DkvStage s0, s1;   /* distinct objects: a read of one never waits for DMA into the other */
    __shared__ uint4 parked[DKV_WAVES][DKV_PARKED][WAVE];   /* the operands the registers do not hold */
    const FaBlock fb = fa_block_order();
    const int seg = fb.seg, h = fb.h;
    const long long start = a.cu[seg];
    const int seglen = a.cu[seg + 1] - a.cu[seg];
    const int k0 = fb.rank * DKV_KEYS;          /* the most query blocks first */
    if (seglen <= 0 || k0 >= seglen) return;
    const int t = threadIdx.x, lane = t & (WAVE - 1), hf = lane >> 5, c = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);   /* in a scalar register, as are the bounds made of it */
    const int kw = k0 + wave * 32;              /* the wave's first key */
    const bool active = kw < seglen;
    const int key = kw + c;

    /* the wave's K and V as B operands: lane (hf, c) holds dims 16 cc + 8 hf .. +7 of key c */
    bf16x8 kb_[8], vb_[8];
    {
        const int n = active ? min(32, seglen - kw) : 0;
        const Rsrc rk = rows_rsrc(a.k, start + kw, a.k_stride, h, n), rv = rows_rsrc(a.v, start + kw, a.v_stride, h, n);
#pragma unroll
        for (int cc = 0; cc < 8; cc++) {
            kb_[cc] = __builtin_bit_cast(bf16x8, bload(rk, (int)((c * a.k_stride + cc * 16 + hf * 8) * 2)));
            vb_[cc] = __builtin_bit_cast(bf16x8, bload(rv, (int)((c * a.v_stride + cc * 16 + hf * 8) * 2)));
        }
        parked[wave][0][lane] = __builtin_bit_cast(uint4, kb_[7]);
        parked[wave][1][lane] = __builtin_bit_cast(uint4, vb_[6]);
        parked[wave][2][lane] = __builtin_bit_cast(uint4, vb_[7]);
    }
    const auto unpark = [&](int i) { return __builtin_bit_cast(bf16x8, parked[wave][i][lane]); };
    f32x16 dk[4], dv[4];
#pragma unroll
    for (int d = 0; d < 4; d++)
#pragma unroll
        for (int i = 0; i < 16; i++) dk[d][i] = dv[d][i] = 0.0f;

    const int qhi = a.window >= 0 ? min(seglen - 1, k0 + DKV_KEYS - 1 + a.window) : seglen - 1;
    /* query block qbk + 1 (Q and dO by LDS DMA, the row statistics through registers) is fetched into the other stage
     * while block qbk is computed; the barrier after the compute makes it visible and frees the one just read */
    float rl = 0.0f, rd = 0.0f;
    const float inv_scale = FA_LOG2E / a.scale_log2;
    auto fetch = [&](int qbk, DkvStage &stg) {
        const int qs = qbk * FA_BN, nq = min(FA_BN, seglen - qs);
        int ln = lane;
        asm volatile("" : "+v"(ln));   /* the DMA's addresses are made here, not held across the loop */
        tile_dma<DKV_WAVES>(a.q, start + qs, a.q_stride, h, nq, stg.q, wave, ln);
        tile_dma<DKV_WAVES>(a.dout, start + qs, a.do_stride, h, nq, stg.dout, wave, ln);
        if (wave == 0) {
            const long long row0 = start + qs;
            const Rsrc rs = make_rsrc(a.lse + (long long)h * a.lse_stride + row0, (unsigned)nq * 4);
            const Rsrc rr = make_rsrc(a.dpsum + row0 * a.H + h, (unsigned)((nq - 1) * a.H + 1) * 4);
            rl = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, ln * 4, 0, 0));
            rd = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rr, ln * a.H * 4, 0, 0));
        }
    };
    auto put_stats = [&](int qbk, DkvStage &stg) {
        if (wave == 0) {
            stg.nlse[lane] = qbk * FA_BN + lane < seglen ? -rl * inv_scale : -INFINITY;
            stg.nd[lane] = -rd;   /* rows past the segment: 0 */
        }
    };
    uint32_t rat = rows_at(lane), tat = tr_at(lane);
    auto compute = [&](int qbk, const DkvStage &s) {
        if (!active) return;
        const int qs = qbk * FA_BN;
#pragma unroll
        for (int qt = 0; qt < 2; qt++) {
            asm volatile("" : "+v"(rat), "+v"(tat));   /* operand addresses are made here, not held across the loop */
            const int q0 = qs + 32 * qt, q1 = q0 + 31, kw1 = kw + 31;
            if (kw > q1 || q0 >= seglen || (a.window >= 0 && q0 - kw1 > a.window)) continue;   /* no row sees the keys */
            const bool interior = kw1 <= q0 && q1 < seglen && kw1 < seglen && (a.window < 0 || q1 - kw <= a.window);
            /* the products start from the rows' statistics (rows q0 + 8 j + 4 hf + i in registers 4 j + i): S - lse / scale,
             * dP - D. The groups keep four operands ahead of their products; two to four measured the same, six 3 % slower,
             * and the dV and dK products' first operands read ahead of the exponentials spilled 20 registers (+ 20 %). */
            f32x16 sc, dp;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const f32x4 l4 = *reinterpret_cast<const f32x4 *>(&s.nlse[32 * qt + 8 * j + 4 * hf]);
#pragma unroll
                for (int i = 0; i < 4; i++) sc[4 * j + i] = l4[i];
            }
#pragma unroll
            for (int cc = 0; cc < 8; cc++)
                sc = mfma32x32x16(rows_operand32(s.q, rat, qt, cc), cc < 7 ? kb_[cc] : unpark(0), sc);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const f32x4 d4 = *reinterpret_cast<const f32x4 *>(&s.nd[32 * qt + 8 * j + 4 * hf]);
#pragma unroll
                for (int i = 0; i < 4; i++) dp[4 * j + i] = d4[i];
            }
#pragma unroll
            for (int cc = 0; cc < 8; cc++)
                dp = mfma32x32x16(rows_operand32(s.dout, rat, qt, cc), cc < 6 ? vb_[cc] : unpark(cc - 5), dp);
            __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);   /* S's statistics, four operands */
#pragma unroll
            for (int m = 0; m < 16; m++) {   /* product m, then the reads of product m + 4: its row operand, a parked one */
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (m == 4) __builtin_amdgcn_sched_group_barrier(0x100, 5, 0);   /* dP's statistics with its first */
                else if (m == 3 || m == 10 || m == 11) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
                else if (m < 12) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
            bf16x8 pb[2], db[2];
            /* P and dS of the lane's 16 (key, row) pairs; only a tile on the diagonal, the window edge or the segment end
             * tests each pair (interior is uniform over the wave: one scalar branch) */
            auto stats = [&](bool masked) {
#pragma unroll
                for (int j = 0; j < 4; j++)
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const float e = __builtin_amdgcn_exp2f(sc[4 * j + i] * a.scale_log2);
                        const float p = !masked || visible(key, q0 + 8 * j + 4 * hf + i, seglen, a.window) ? e : 0.0f;
                        const float ds = p * dp[4 * j + i];
                        pb[j >> 1][(j & 1) * 4 + i] = (__bf16)p;
                        db[j >> 1][(j & 1) * 4 + i] = (__bf16)ds;
                    }
            };
            if (interior)
                stats(false);
            else
                stats(true);
#pragma unroll
            for (int s2 = 0; s2 < 2; s2++)
#pragma unroll
                for (int d = 0; d < 4; d++) {
                    dv[d] = mfma32x32x16(tr_operand32(s.dout, tat, d, 32 * qt + 16 * s2), pb[s2], dv[d]);
                    dk[d] = mfma32x32x16(tr_operand32(s.q, tat, d, 32 * qt + 16 * s2), db[s2], dk[d]);
                }
            __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);   /* two steps' operands ahead of their products */
#pragma unroll
            for (int st = 0; st < 8; st++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
                if (st < 6) __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
            }
        }
    };
    const int qb_lo = k0 / FA_BN, qb_hi = qhi / FA_BN;
    fetch(qb_lo, s0);
    put_stats(qb_lo, s0);
    __syncthreads();
    for (int qbk = qb_lo; qbk <= qb_hi; qbk += 2) {
        if (qbk + 1 <= qb_hi) fetch(qbk + 1, s1);
        compute(qbk, s0);
        if (qbk + 1 <= qb_hi) put_stats(qbk + 1, s1);
        __syncthreads();
        if (qbk + 1 > qb_hi) break;
        if (qbk + 2 <= qb_hi) fetch(qbk + 2, s0);
        compute(qbk + 1, s1);
        if (qbk + 2 <= qb_hi) put_stats(qbk + 2, s0);
        __syncthreads();
    }
    if (!active || key >= seglen) return;
    /* dK^T, dV^T tile d: lane (hf, c) holds dims 32 d + 8 j + 4 hf .. +3 of key c in registers 4 j .. + 3 */
    uint16_t *pk = a.dk + (start + key) * a.dk_stride + (long long)h * HEAD_DIM + 4 * hf;
    uint16_t *pv = a.dv + (start + key) * a.dv_stride + (long long)h * HEAD_DIM + 4 * hf;
#pragma unroll
    for (int d = 0; d < 4; d++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            store4(pk + d * 32 + 8 * j, f32x4{dk[d][4 * j], dk[d][4 * j + 1], dk[d][4 * j + 2], dk[d][4 * j + 3]}, a.scale);
            store4(pv + d * 32 + 8 * j, f32x4{dv[d][4 * j], dv[d][4 * j + 1], dv[d][4 * j + 2], dv[d][4 * j + 3]}, 1.0f);
        }
}

struct DqStage {
    uint16_t k[FA_BN * HEAD_DIM], v[FA_BN * HEAD_DIM];   /* k_lds layout; K^T read transposed */
};

/* dQ of 128 queries: as the forward, S^T = K Q^T and dP^T = V dO^T with queries as columns, so dS^T feeds
 * dQ^T += K^T dS^T as the B operand with K^T read from a transposed LDS tile. Bound as the forward is. 32 x 32 products
 * read the same operand bytes as two 16-wide tiles a wave did; they win by the lse and D they start from (a column's two
 * scalars, so P and dS are one multiplication each) and by skipping 32-key tiles no row sees. The backward's share
 * of 1 x 8,192 tokens x 6 heads: 499 -> 468 us, 32 x 2,048 x 6 800 -> 781, 8 x 2,048 x 10 with window 512 206 -> 196. */
__global__ void __launch_bounds__(FA_THREADS, 2) flash_bwd_dq_kernel(FlashBwd a) {
    __shared__ DqStage s0, s1;   /* distinct objects: a read of one never waits for DMA into the other */
    const FaBlock fb = fa_block_order();
    const int seg = fb.seg, h = fb.h;
    const long long start = a.cu[seg];
    const int seglen = a.cu[seg + 1] - a.cu[seg];
    const int tile = (int)gridDim.x - 1 - fb.rank;
    const int qa = tile * FA_BM;
    if (seglen <= 0 || qa >= seglen) return;
    const int t = threadIdx.x, lane = t & (WAVE - 1), hf = lane >> 5, c = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);   /* in a scalar register, as are the bounds made of it */
    const int qb = min(qa + FA_BM, seglen) - 1;
    const int q0 = qa + wave * 32;
    const bool active = q0 < seglen;
    const int qw1 = min(q0 + 31, seglen - 1);

    /* queries and dO as B operands (lane (hf, c): dims 16 cc + 8 hf .. +7 of row c); the column's -lse / scale and -D,
     * from which its S and dP products start */
    bf16x8 qb_[8], ob_[8];
    float nlse, nd;
    {
        const int n = active ? min(32, seglen - q0) : 0;
        const Rsrc rq = rows_rsrc(a.q, start + q0, a.q_stride, h, n), ro = rows_rsrc(a.dout, start + q0, a.do_stride, h, n);
#pragma unroll
        for (int cc = 0; cc < 8; cc++) {
            qb_[cc] = __builtin_bit_cast(bf16x8, bload(rq, (int)((c * a.q_stride + cc * 16 + hf * 8) * 2)));
            ob_[cc] = __builtin_bit_cast(bf16x8, bload(ro, (int)((c * a.do_stride + cc * 16 + hf * 8) * 2)));
        }
        const bool ok = c < n;
        nlse = ok ? a.lse[(long long)h * a.lse_stride + start + q0 + c] * (-FA_LOG2E / a.scale_log2) : -INFINITY;
        nd = ok ? -a.dpsum[(start + q0 + c) * a.H + h] : 0.0f;
    }
    f32x16 dq[4];
#pragma unroll
    for (int d = 0; d < 4; d++)
#pragma unroll
        for (int i = 0; i < 16; i++) dq[d][i] = 0.0f;

    const int klo = a.window >= 0 ? max(0, qa - a.window) : 0;
    /* key block kb + 1 (K and V by LDS DMA) is fetched into the other stage while block kb is computed */
    auto fetch = [&](int kb, DqStage &stg) {
        const int nk = min(FA_BN, seglen - kb * FA_BN);
        tile_dma(a.k, start + kb * FA_BN, a.k_stride, h, nk, stg.k, wave, lane);
        tile_dma(a.v, start + kb * FA_BN, a.v_stride, h, nk, stg.v, wave, lane);
    };
    uint32_t rat = rows_at(lane), tat = tr_at(lane);
    auto compute = [&](int kb, const DqStage &s) {
        if (!active) return;
#pragma unroll
        for (int kt = 0; kt < 2; kt++) {
            asm volatile("" : "+v"(rat), "+v"(tat));   /* operand addresses are made here, not held across the loop */
            const int k0 = kb * FA_BN + 32 * kt, k1 = k0 + 31;
            if (k0 > qw1 || (a.window >= 0 && q0 - k1 > a.window)) continue;   /* no row sees the keys */
            const bool interior = k1 <= q0 && k1 < seglen && (a.window < 0 || qw1 - k0 <= a.window);
            f32x16 sc, dp;
#pragma unroll
            for (int i = 0; i < 16; i++) { sc[i] = nlse; dp[i] = nd; }
#pragma unroll
            for (int cc = 0; cc < 8; cc++) {
                sc = mfma32x32x16(rows_operand32(s.k, rat, kt, cc), qb_[cc], sc);
                dp = mfma32x32x16(rows_operand32(s.v, rat, kt, cc), ob_[cc], dp);
            }
            products_in_order<16, 1>();
            /* lane (hf, c): query column c, keys k0 + 8 j + 4 hf + i; only a tile on the diagonal, the window edge or the
             * segment end tests each pair (interior is uniform: one scalar branch) */
            bf16x8 db[2];
            auto pds = [&](bool masked) {
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const float e = __builtin_amdgcn_exp2f(sc[i] * a.scale_log2);
                    const float p =
                        !masked || visible(k0 + 8 * (i >> 2) + 4 * hf + (i & 3), q0 + c, seglen, a.window) ? e : 0.0f;
                    db[i >> 3][i & 7] = (__bf16)(p * dp[i]);
                }
            };
            if (interior)
                pds(false);
            else
                pds(true);
#pragma unroll
            for (int s2 = 0; s2 < 2; s2++)
#pragma unroll
                for (int d = 0; d < 4; d++)
                    dq[d] = mfma32x32x16(tr_operand32(s.k, tat, d, 32 * kt + 16 * s2), db[s2], dq[d]);
            products_in_order<8, 2>();
        }
    };
    const int kb_lo = klo / FA_BN, kb_hi = qb / FA_BN;
    fetch(kb_lo, s0);
    __syncthreads();
    for (int kb = kb_lo; kb <= kb_hi; kb += 2) {
        if (kb + 1 <= kb_hi) fetch(kb + 1, s1);
        compute(kb, s0);
        __syncthreads();
        if (kb + 1 > kb_hi) break;
        if (kb + 2 <= kb_hi) fetch(kb + 2, s0);
        compute(kb + 1, s1);
        __syncthreads();
    }
    if (!active || q0 + c >= seglen) return;
    uint16_t *p = a.dq + (start + q0 + c) * a.dq_stride + (long long)h * HEAD_DIM + 4 * hf;
#pragma unroll
    for (int d = 0; d < 4; d++)
#pragma unroll
        for (int j = 0; j < 4; j++)
            store4(p + d * 32 + 8 * j, f32x4{dq[d][4 * j], dq[d][4 * j + 1], dq[d][4 * j + 2], dq[d][4 * j + 3]}, a.scale);
}

/* D[row][h] = sum_d dO . O in fp32, bound by HBM (512 bytes a row): 16 lanes a (row, head), eight consecutive dims a lane
 * by 16-byte loads (4-byte aligned), the lanes' sums by the fixed butterfly. 65,536 tokens of 6 heads 31 us; a wave a row
 * with 4 bytes a lane took 62. */
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

__global__ void __launch_bounds__(256) flash_bwd_rows_kernel(const uint16_t *out, long long o_stride,
                                                             const uint16_t *dout, long long do_stride, long long n,
                                                             int H, float *dpsum) {
    const long long w = (long long)blockIdx.x * 16 + (threadIdx.x >> 4);
    if (w >= n) return;   /* whole 16-lane groups */
    const int i = threadIdx.x & 15;
    const long long row = n < (1LL << 31) ? (long long)((unsigned)w / (unsigned)H) : w / H;
    const int h = (int)(w - row * H);
    const u32x4_a4 o = *reinterpret_cast<const u32x4_a4 *>(out + row * o_stride + (long long)h * HEAD_DIM + 8 * i);
    const u32x4_a4 d = *reinterpret_cast<const u32x4_a4 *>(dout + row * do_stride + (long long)h * HEAD_DIM + 8 * i);
    float v = 0.0f;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        v = __builtin_fmaf(__uint_as_float(o[k] << 16), __uint_as_float(d[k] << 16), v);
        v = __builtin_fmaf(__uint_as_float(o[k] & 0xFFFF0000u), __uint_as_float(d[k] & 0xFFFF0000u), v);
    }
    v = v + lane_xor_dpp<8>(v);
    v = v + lane_xor_dpp<4>(v);
    v = v + lane_xor_dpp<2>(v);
    v = v + lane_xor_dpp<1>(v);
    if (i == 0) dpsum[w] = v;
}

}  // namespace
}  // namespace nc

using namespace nc;

extern "C" int nc_flash_attn_fwd(const void *q, const void *k, const void *v, long long q_stride, long long k_stride,
                                 long long v_stride, const int32_t *cu_seqlens, int segments, int max_seqlen,
                                 int heads, int window, float softmax_scale, void *out, float *lse,
                                 long long lse_stride, void *stream) {
    if (segments < 0 || max_seqlen < 0 || heads < 1 || heads > 65535 || segments > 65535 || lse_stride < 0 ||
        !(softmax_scale > 0.0f))
        return NC_ERR_SHAPE;
    if (segments == 0 || max_seqlen == 0) return NC_OK;
    if (!q || !k || !v || !cu_seqlens || !out || !lse) return NC_ERR_NULL;
    const long long row = (long long)heads * HEAD_DIM;
    if (q_stride < row || k_stride < row || v_stride < row || q_stride % 8 || k_stride % 8 || v_stride % 8 ||
        ((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out) & 15)
        return NC_ERR_SHAPE;
    /* a block of 64 rows of one head is one buffer descriptor with 32-bit signed offsets */
    if ((63 * max(max(q_stride, k_stride), v_stride) + HEAD_DIM) * 2 >= 0x7FFFFFFFLL) return NC_ERR_SHAPE;
    FlashFwd a;
    a.q = (const uint16_t *)q; a.k = (const uint16_t *)k; a.v = (const uint16_t *)v;
    a.q_stride = q_stride; a.k_stride = k_stride; a.v_stride = v_stride;
    a.cu = cu_seqlens; a.segments = segments; a.H = heads; a.window = window < 0 ? -1 : window;
    a.scale_log2 = softmax_scale * FA_LOG2E;
    a.out = (uint16_t *)out; a.lse = lse; a.lse_stride = lse_stride;
    const dim3 grid((unsigned)((max_seqlen + FA_BM - 1) / FA_BM), (unsigned)segments, (unsigned)heads);
    hipLaunchKernelGGL(flash_fwd_kernel, grid, dim3(FA_THREADS), 0, (hipStream_t)stream, a);
    return (int)hipGetLastError();
}

extern "C" int nc_flash_attn_bwd_rows(const void *out, long long o_stride, const void *dout, long long do_stride,
                                      long long total, int heads, float *dpsum, void *stream) {
    if (total < 0 || heads < 1 || o_stride < (long long)heads * HEAD_DIM || do_stride < (long long)heads * HEAD_DIM ||
        o_stride % 2 || do_stride % 2)
        return NC_ERR_SHAPE;
    if (total == 0) return NC_OK;
    if (!out || !dout || !dpsum) return NC_ERR_NULL;
    if (((uintptr_t)out | (uintptr_t)dout) & 3) return NC_ERR_SHAPE;
    const long long n = total * heads;
    hipLaunchKernelGGL(flash_bwd_rows_kernel, dim3((unsigned)((n + 15) / 16)), dim3(256), 0, (hipStream_t)stream,
                       (const uint16_t *)out, o_stride, (const uint16_t *)dout, do_stride, n, heads, dpsum);
    return (int)hipGetLastError();
}

extern "C" int nc_flash_attn_bwd(const void *q, const void *k, const void *v, const void *dout, long long q_stride,
                                 long long k_stride, long long v_stride, long long do_stride, const float *lse,
                                 long long lse_stride, const float *dpsum, const int32_t *cu_seqlens, int segments,
                                 int max_seqlen, int heads, int window, float softmax_scale, void *dq, void *dk,
                                 void *dv, long long dq_stride, long long dk_stride, long long dv_stride,
                                 void *stream) {
    if (segments < 0 || max_seqlen < 0 || heads < 1 || heads > 65535 || segments > 65535 || lse_stride < 0 ||
        !(softmax_scale > 0.0f))
        return NC_ERR_SHAPE;
    if (segments == 0 || max_seqlen == 0) return NC_OK;
    if (!q || !k || !v || !dout || !lse || !dpsum || !cu_seqlens || !dq || !dk || !dv) return NC_ERR_NULL;
    const long long row = (long long)heads * HEAD_DIM;
    const long long strides[] = {q_stride, k_stride, v_stride, do_stride, dq_stride, dk_stride, dv_stride};
    long long widest = 0;
    for (long long st : strides) {
        if (st < row || st % 8) return NC_ERR_SHAPE;
        widest = max(widest, st);
    }
    if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)dout | (uintptr_t)dq | (uintptr_t)dk | (uintptr_t)dv) & 15)
        return NC_ERR_SHAPE;
    if ((63 * widest + HEAD_DIM) * 2 >= 0x7FFFFFFFLL) return NC_ERR_SHAPE;
    FlashBwd a;
    a.q = (const uint16_t *)q; a.k = (const uint16_t *)k; a.v = (const uint16_t *)v; a.dout = (const uint16_t *)dout;
    a.q_stride = q_stride; a.k_stride = k_stride; a.v_stride = v_stride; a.do_stride = do_stride;
    a.lse = lse; a.lse_stride = lse_stride; a.dpsum = dpsum;
    a.cu = cu_seqlens; a.segments = segments; a.H = heads; a.window = window < 0 ? -1 : window;
    /* the kernels divide lse by the exponent's scale: kept where that quotient is finite; below, scale S vanishes beside
     * lse */
    a.scale = softmax_scale; a.scale_log2 = fmaxf(softmax_scale, 0x1p-116f) * FA_LOG2E;
    a.dq = (uint16_t *)dq; a.dk = (uint16_t *)dk; a.dv = (uint16_t *)dv;
    a.dq_stride = dq_stride; a.dk_stride = dk_stride; a.dv_stride = dv_stride;
    hipLaunchKernelGGL(flash_bwd_dkv_kernel, dim3((unsigned)((max_seqlen + DKV_KEYS - 1) / DKV_KEYS),
                                                  (unsigned)segments, (unsigned)heads),
                       dim3(64 * DKV_WAVES), 0, (hipStream_t)stream, a);
    hipLaunchKernelGGL(flash_bwd_dq_kernel, dim3((unsigned)((max_seqlen + FA_BM - 1) / FA_BM), (unsigned)segments,
                                                 (unsigned)heads),
                       dim3(FA_THREADS), 0, (hipStream_t)stream, a);
    return (int)hipGetLastError();
}
