/*
 * Cache append for the fp8 KV path on gfx950: the fused q/k RMS norm + gain + -theta rotation, the
 * per-(token, KV head) absmax e4m3fn quantizer and the paged store; plus the training-form q/k prologue
 * (the reference's qkp_forward) on the same row math.
 *
 * Four (token, head) rows a wave, 16 lanes a row. The row math (nc_row.h) gives the same bits as the fused decode
 * step's, which appends the step's token inside the attention kernel.
 */
#include "nc_device.h"
#include "nc_row.h"
#include "nanochat_amd.h"
#include "nc_internal.h"

namespace nc {

struct AppendArgs {
    const uint16_t *k, *v;     /* plain append: [B][T][Hkv][128] at token_stride */
    const uint16_t *qkv;       /* fused append: [B][T][(Hq + 2 Hkv) 128] at token_stride */
    long long token_stride;
    int B, T, Hq, Hkv;
    const int32_t *start_pos, *num_new;
    const int32_t *row0;       /* NULL: sequence b's tokens are rows b T + t; else rows row0[b] + t */
    const float *q_gain, *k_gain, *cos, *sin;
    int rope_len;
    uint16_t *q_out;           /* [rows][Hq][128] */
    const int32_t *block_table;
    const int32_t *seq_slot;   /* NULL, or sequence b's block-table row (the decoder's prefill runs) */
    /* value embeddings (fused append, NULL ve: none): v += 2 sigmoid(ve_gate[head] . h) ve[tokens[token]] */
    const uint16_t *ve_h, *ve;  /* h: [rows][C] the layer's normed input; ve: [vocab][C] */
    const float *ve_gate;       /* [Hkv][C] */
    const int32_t *ve_tokens;   /* [rows] */
    int C;
    int max_pages;
    uint8_t *k_pages, *v_pages;
    float *kv_scale;          /* [num_pages][Hkv][2][16]: K scales, then V scales */
    int num_pages;
    int pages_per_seq;        /* grid x = B pages_per_seq: the most cache pages T positions can touch */
};

/* Cache pages a run of T positions can touch: (T - 1) / 16 + 1 when aligned, one more when not. */
static inline int append_pages_per_seq(int T) { return (T + PAGE - 2) / PAGE + 1; }

/* Grid: x = (sequence b, k-th cache page its new positions touch), y = head groups; block = 4 waves.
 * The new positions of b are [max(start, 0), start + min(T, num_new[b])), cut at rope_len when FUSED (the rest are
 * skipped, as are all of b's positions on a page past max_pages or whose table entry lies outside the pool). The
 * work-group takes those of them on page k: slots [s_lo, s_hi) of that page. Rows are computed four a wave, 16 lanes
 * a row (nc_row.h's 16-lane form, the same bits as the one-row-a-wave form of the fused
 * decode step), wave w slots 4 w .. 4 w + 3.
 * y < Hkv: KV head y. The k rows (norm and rotation when FUSED, then the quantizer) and the v rows (the value-embedding
 * mix when given, then the quantizer) leave their codes in an LDS image of the page in the cache's layout. The work-group
 * then stores the image with one 16-byte store a lane; a K block holds one slot, a V block four (slots 4 g .. 4 g + 3),
 * and a V block holding slots outside [s_lo, s_hi) is stored byte by byte, so the page's other slots keep their bytes.
 * The 16 scales of K and of V go out the same way.
 * y >= Hkv (FUSED only): q heads 4 (y - Hkv) .. + 3 of the page's slots, normed and rotated into q_out; a wave reads its
 * slots' rotation once for the four.
 * It is bound by the chain each work-group begins with (position, page, rows) more than by HBM: 46 MB in 12.9 us (12.4 at best)
 * at 8 x 512 tokens of 16 / 4 heads (13.2 with eight 2-byte accesses a row and lane), 75 MB in 21.8 us at 3 x 1,501 tokens of
 * 13 / 13 heads (22.4); with value embeddings, 6,594 rows of 6 heads, C = 768, 36 -> 24 us. Four KV heads a work-group, one
 * chain for all, left too few of them: 17 us, 25 us and 37 us. */
constexpr int Q_GROUP = 4;   /* q heads a work-group */

template <bool FUSED>
__global__ void __launch_bounds__(256) append_kernel(AppendArgs a) {
    __shared__ __align__(16) uint8_t img[2][PAGE_BYTES];
    __shared__ float img_scale[2][PAGE];
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x >> 6;
    const int r = lane >> 4, i = lane & 15;   /* the lane's row of the wave's four, its place in the row */
    const int b = blockIdx.x / a.pages_per_seq, k = blockIdx.x % a.pages_per_seq;
    const int sp = a.start_pos[b];
    const int n = a.num_new ? min(a.num_new[b], a.T) : a.T;
    const long long lo = max(sp, 0);
    long long hi = (long long)sp + n;
    if (FUSED && hi > a.rope_len) hi = a.rope_len;
    if (lo >= hi) return;
    const long long lp = lo / PAGE + k, pg0 = lp * PAGE;
    const int s_lo = (int)(max(lo, pg0) - pg0), s_hi = (int)(min(hi, pg0 + PAGE) - pg0);
    if (s_lo >= s_hi) return;
    const long long tok_at = (a.row0 ? (long long)a.row0[b] : (long long)b * a.T) - sp;   /* + position = row */
    const int slot = 4 * wave + r;
    const bool live = slot >= s_lo && slot < s_hi;   /* rows of other slots compute a new one and store nothing */
    const long long p = pg0 + min(max(slot, s_lo), s_hi - 1), tok = tok_at + p;

    if (FUSED && (int)blockIdx.y >= a.Hkv) {
        const int h0 = Q_GROUP * ((int)blockIdx.y - a.Hkv);
        const uint16_t *row = a.qkv + tok * a.token_stride + h0 * HEAD_DIM;
        uint4 raw[Q_GROUP];
        float g[8], c[4], s[4];
#pragma unroll
        for (int j = 0; j < Q_GROUP; j++)
            if (h0 + j < a.Hq) raw[j] = load_row16(row + j * HEAD_DIM, i);
        load4_f32(a.cos + p * HALF + 4 * i, c);
        load4_f32(a.sin + p * HALF + 4 * i, s);
        load_gain16(a.q_gain, i, g);
        uint16_t *q = a.q_out + (tok * a.Hq + h0) * HEAD_DIM;
#pragma unroll
        for (int j = 0; j < Q_GROUP; j++) {
            if (h0 + j >= a.Hq) break;
            float x[8], y[8];
            unpack8(raw[j], x);
            norm_rope16(x, g, c, s, y);
            if (live) store_row16(q + j * HEAD_DIM, i, y);
        }
        return;
    }

    const int kvh = blockIdx.y;
    if (lp >= a.max_pages) return;
    const int trow = a.seq_slot ? a.seq_slot[b] : b;
    const int page = a.block_table[(long long)trow * a.max_pages + lp];
    if (page < 0 || page >= a.num_pages) return;
    const long long at = (long long)page * a.Hkv + kvh;

    const uint16_t *kx = FUSED ? a.qkv + tok * a.token_stride + (a.Hq + kvh) * HEAD_DIM
                               : a.k + tok * a.token_stride + kvh * HEAD_DIM;
    const uint16_t *vx = FUSED ? a.qkv + tok * a.token_stride + (a.Hq + a.Hkv + kvh) * HEAD_DIM
                               : a.v + tok * a.token_stride + kvh * HEAD_DIM;
    const uint4 kraw = load_row16(kx, i), vraw = load_row16(vx, i);
    float x[8];
    unpack8(kraw, x);
    if (FUSED) {
        float g[8], c[4], s[4], y[8];
        load4_f32(a.cos + p * HALF + 4 * i, c);
        load4_f32(a.sin + p * HALF + 4 * i, s);
        load_gain16(a.k_gain, i, g);
        norm_rope16(x, g, c, s, y);
        unpack8(pack8(y), x);
    }
    uint32_t code[2];
    float scale = quantize16(x, code);
    if (live) {
        *reinterpret_cast<uint32_t *>(&img[0][k_page_offset(slot, 4 * i)]) = code[0];
        *reinterpret_cast<uint32_t *>(&img[0][k_page_offset(slot, HALF + 4 * i)]) = code[1];
        if (i == 0) img_scale[0][slot] = scale;
    }
    unpack8(vraw, x);
    if (FUSED && a.ve)
        ve_mix16(a.ve_h + tok * a.C, a.ve_gate + (long long)kvh * a.C, a.C,
                 a.ve + (long long)a.ve_tokens[tok] * a.C + kvh * HEAD_DIM, i, x);
    scale = quantize16(x, code);
    if (live) {
#pragma unroll
        for (int e = 0; e < 8; e++)
            img[1][v_page_offset(slot, (e < 4 ? 4 * i : HALF + 4 * i) + (e & 3))] = (uint8_t)(code[e >> 2] >> (8 * (e & 3)));
        if (i == 0) img_scale[1][slot] = scale;
    }
    __syncthreads();

    const int t = threadIdx.x, blk = t & 127, kind = t >> 7;   /* kind 0: K block, 1: V block */
    uint8_t *dst = (kind ? a.v_pages : a.k_pages) + at * PAGE_BYTES + blk * 16;
    const uint8_t *src = img[kind] + blk * 16;
    const int s_first = kind ? 4 * ((blk >> 4) & 3) : (blk & 15), s_count = kind ? 4 : 1;
    if (s_first >= s_lo && s_first + s_count <= s_hi) {
        *reinterpret_cast<uint4 *>(dst) = *reinterpret_cast<const uint4 *>(src);
    } else if (kind && s_first < s_hi && s_first + s_count > s_lo) {
#pragma unroll
        for (int e = 0; e < 16; e++) {   /* byte e holds slot s_first + e % 4 */
            const int sl = s_first + (e & 3);
            if (sl >= s_lo && sl < s_hi) dst[e] = src[e];
        }
    }
    if (t < 2 * PAGE) {
        const int sl = t & (PAGE - 1), kv = t >> 4;
        if (sl >= s_lo && sl < s_hi) a.kv_scale[(at * 2 + kv) * PAGE + sl] = img_scale[kv][sl];
    }
}

/* The training-form prologue (reference model/kernels/qk_prologue.cu:8-32) of q's and k's [tokens][H] rows: input
 * token stride 3 H 128, output contiguous, position p % T for token p.
 *
 * Both directions are bound by HBM (forward: 2 x 256 bytes a row; backward: 3 x 256). 16 lanes take a row (nc_row.h's
 * form), a 16-lane group QK_HEADS heads of one token, so an access is 8 or 16 bytes a lane, the rotation is read once for
 * QK_HEADS rows and all of a group's rows are in flight together. Against one row a wave with 2-byte accesses, 65,536
 * tokens of 6 heads: forward 179 -> 87 us (4.6 TB/s), backward 242 -> 115 us (5.2 TB/s); a copy, which reads as much as it
 * writes, reaches 4.8.
 * QK_HEADS divides the 6 heads of the small model and is the same for every count, a group's last places being empty where
 * it does not divide. 65,536 tokens, caches cold, forward / backward in us with two, three and four heads a group: 1 head
 * 25 / 42 each; 4 heads 79 / 119, 86 / 126, 77 / 121; 6 heads 101 / 154, 101 / 156, 112 / 162; 10 heads 150 / 228,
 * 161 / 238, 149 / 237; 16 heads 229 / 347, 233 / 352, 220 / 352. */
constexpr int QK_HEADS = 3;
static int qk_head_chunks(int H) { return (H + QK_HEADS - 1) / QK_HEADS; }

/* Grid x = 16-token blocks times the head chunks of q then of k (chunk fastest), 256 threads. Indexes fit 32 bits: a row
 * takes 768 bytes of memory or more. */
__global__ void __launch_bounds__(256) qkp_forward_kernel(const uint16_t *q, const uint16_t *k, const float *gq,
                                                          const float *gk, uint16_t *qo, uint16_t *ko,
                                                          const float *cos, const float *sin, long long tokens, int H,
                                                          int T) {
    const int i = threadIdx.x & 15, chunks = (H + QK_HEADS - 1) / QK_HEADS;
    const int block = blockIdx.x / (2 * chunks), chunk = blockIdx.x - block * 2 * chunks;
    const long long p = (long long)block * 16 + (threadIdx.x >> 4);
    if (p >= tokens) return;   /* whole 16-lane groups */
    const bool isq = chunk < chunks;
    const int h0 = (chunk - (isq ? 0 : chunks)) * QK_HEADS;
    const uint16_t *x = (isq ? q : k) + (p * 3 * H + h0) * HEAD_DIM;
    uint16_t *y = (isq ? qo : ko) + (p * H + h0) * HEAD_DIM;
    const long long tab = (long long)((unsigned)p % (unsigned)T) * HALF + 4 * i;
    uint4 raw[QK_HEADS];
    float g[8], c[4], s[4];
#pragma unroll
    for (int j = 0; j < QK_HEADS; j++)
        if (h0 + j < H) raw[j] = load_row16(x + j * HEAD_DIM, i);
    load4_f32(cos + tab, c);
    load4_f32(sin + tab, s);
    load_gain16(isq ? gq : gk, i, g);
#pragma unroll
    for (int j = 0; j < QK_HEADS; j++) {
        if (h0 + j >= H) break;
        float xr[8], yr[8];
        unpack8(raw[j], xr);
        norm_rope16(xr, g, c, s, yr);
        store_row16(y + j * HEAD_DIM, i, yr);
    }
}

/* The prologue's backward (reference model/kernels/qk_prologue.cu:36-90): per (token, head) row, recomputing n = x r;
 * the rotation's transpose gives dm (dm1 = dy1 c - dy2 s, dm2 = dy1 s + dy2 c); dn = dm g; dx = r (dn - n b),
 * b = sum(dn n) / 128 (the butterfly); the gain gradient sum_rows dm n accumulates per lane in row order. Grid:
 * QKB_BLOCKS blocks per tensor (q's, then k's); 16-lane group w of a tensor's QKB_GROUPS takes the (token, head chunk)
 * units w, w + QKB_GROUPS, ...; each block writes its partial [128] (its groups added in order). */
constexpr int QKB_BLOCKS = 512;   /* fixed, so the gain gradient's summation order is fixed */
constexpr int QKB_GROUPS = QKB_BLOCKS * 16;

__global__ void __launch_bounds__(256) qkp_backward_kernel(const uint16_t *q, const uint16_t *k, const float *gq,
                                                           const float *gk, const uint16_t *dqo, const uint16_t *dko,
                                                           uint16_t *dq, uint16_t *dk, const float *cos,
                                                           const float *sin, float *part, long long tokens, int H,
                                                           int T) {
    __shared__ float gpart[16][HEAD_DIM];
    const int i = threadIdx.x & 15, grp = threadIdx.x >> 4;
    const bool isq = blockIdx.x < QKB_BLOCKS;
    const uint16_t *xin = isq ? q : k, *dyin = isq ? dqo : dko;
    uint16_t *dxout = isq ? dq : dk;
    const unsigned chunks = (H + QK_HEADS - 1) / QK_HEADS;
    float g[8], acc[8];
    load_gain16(isq ? gq : gk, i, g);
#pragma unroll
    for (int e = 0; e < 8; e++) acc[e] = 0.0f;
    const unsigned units = (unsigned)(tokens * chunks);
    for (unsigned u = (isq ? blockIdx.x : blockIdx.x - QKB_BLOCKS) * 16 + grp; u < units; u += QKB_GROUPS) {
        const unsigned t = u / chunks;
        const int h0 = (int)(u - t * chunks) * QK_HEADS;
        const long long at = ((long long)t * 3 * H + h0) * HEAD_DIM, row = ((long long)t * H + h0) * HEAD_DIM;
        const long long tab = (long long)(t % (unsigned)T) * HALF + 4 * i;
        uint4 xraw[QK_HEADS], draw[QK_HEADS];
        float c[4], s[4];
#pragma unroll
        for (int j = 0; j < QK_HEADS; j++)
            if (h0 + j < H) {
                xraw[j] = load_row16(xin + at + j * HEAD_DIM, i);
                draw[j] = load_row16(dyin + row + j * HEAD_DIM, i);
            }
        load4_f32(cos + tab, c);
        load4_f32(sin + tab, s);
#pragma unroll
        for (int j = 0; j < QK_HEADS; j++) {
            if (h0 + j >= H) break;
            float x[8], d[8], n[8], dn[8], prod[4], dx[8];
            unpack8(xraw[j], x);
            unpack8(draw[j], d);
            const float r = rstd16(x);
#pragma unroll
            for (int e = 0; e < 8; e++) n[e] = x[e] * r;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float dm1 = d[e] * c[e] - d[e + 4] * s[e], dm2 = d[e] * s[e] + d[e + 4] * c[e];
                acc[e] = acc[e] + dm1 * n[e];
                acc[e + 4] = acc[e + 4] + dm2 * n[e + 4];
                dn[e] = dm1 * g[e];
                dn[e + 4] = dm2 * g[e + 4];
                prod[e] = dn[e] * n[e] + dn[e + 4] * n[e + 4];
            }
            const float b = lane16_sum(prod) / 128.0f;
#pragma unroll
            for (int e = 0; e < 8; e++) dx[e] = r * (dn[e] - n[e] * b);
            store_row16(dxout + at + j * HEAD_DIM, i, dx);
        }
    }
#pragma unroll
    for (int e = 0; e < 8; e++) gpart[grp][(e < 4 ? 0 : HALF) + 4 * i + (e & 3)] = acc[e];
    __syncthreads();
    if (threadIdx.x < HEAD_DIM) {
        float sum = gpart[0][threadIdx.x];
#pragma unroll
        for (int w = 1; w < 16; w++) sum = sum + gpart[w][threadIdx.x];
        part[(long long)blockIdx.x * HEAD_DIM + threadIdx.x] = sum;
    }
}

/* Grid (2 tensors, HEAD_DIM / 16): the gain gradients of 16 dims from the QKB_BLOCKS partials (reference
 * qk_prologue.cu:92-97). A serial sum of 512 partials is a chain of loads (11 us); here thread (w, d) adds partials
 * 32 w .. 32 w + 31 of dim d, all loads issued together, and the 16 sums are added in order (4 us). */
__global__ void __launch_bounds__(256) qkp_gain_sum_kernel(const float *part, float *dgq, float *dgk) {
    constexpr int PER = QKB_BLOCKS / 16;
    __shared__ float sums[16][16];
    const int d = threadIdx.x & 15, w = threadIdx.x >> 4, dim = blockIdx.y * 16 + d;
    const float *p = part + ((long long)blockIdx.x * QKB_BLOCKS + w * PER) * HEAD_DIM + dim;
    float v[PER], sum = 0.0f;
#pragma unroll
    for (int j = 0; j < PER; j++) v[j] = p[j * HEAD_DIM];
#pragma unroll
    for (int j = 0; j < PER; j++) sum = sum + v[j];
    sums[w][d] = sum;
    __syncthreads();
    if (w) return;
#pragma unroll
    for (int j = 1; j < 16; j++) sum = sum + sums[j][d];
    (blockIdx.x ? dgk : dgq)[dim] = sum;
}

static thread_local int last_error = NC_OK;

static int launch_append(AppendArgs a, bool fused, hipStream_t stream) {
    a.pages_per_seq = append_pages_per_seq(a.T);
    const long long x = (long long)a.B * a.pages_per_seq;
    if (x * 256 >= (1LL << 32)) return NC_ERR_SHAPE;
    const dim3 grid((unsigned)x, (unsigned)(a.Hkv + (fused ? (a.Hq + Q_GROUP - 1) / Q_GROUP : 0)));
    if (fused)
        hipLaunchKernelGGL(append_kernel<true>, grid, dim3(256), 0, stream, a);
    else
        hipLaunchKernelGGL(append_kernel<false>, grid, dim3(256), 0, stream, a);
    return (int)hipGetLastError();
}

/* The fused append for the decoder runtime's prefill: runs of rows, run r being rows row0[r] .. + count[r] - 1 of
 * qkv (token_stride apart), at positions start[r] .. of block-table row seq_slot[r], max_count the longest run; with
 * ve non-NULL, v gets the layer's value embedding. Arguments are checked by the caller. */
int append_runs(const uint16_t *qkv, long long token_stride, int runs, int max_count, const int32_t *row0,
                const int32_t *count, const int32_t *start, const int32_t *seq_slot, int Hq, int Hkv,
                const float *q_gain, const float *k_gain, const float *cos, const float *sin, int rope_len,
                uint16_t *q_out, const int32_t *block_table, int max_pages, uint8_t *k_pages, uint8_t *v_pages,
                float *kv_scale, int num_pages, const uint16_t *ve_h, const uint16_t *ve, const float *ve_gate,
                const int32_t *tokens, int C, hipStream_t stream) {
    if (runs <= 0 || max_count <= 0) return NC_OK;
    AppendArgs a = {};
    a.qkv = qkv;
    a.token_stride = token_stride;
    a.B = runs; a.T = max_count; a.Hq = Hq; a.Hkv = Hkv;
    a.start_pos = start; a.num_new = count; a.row0 = row0; a.seq_slot = seq_slot;
    a.q_gain = q_gain; a.k_gain = k_gain; a.cos = cos; a.sin = sin; a.rope_len = rope_len;
    a.q_out = q_out;
    a.block_table = block_table; a.max_pages = max_pages;
    a.k_pages = k_pages; a.v_pages = v_pages; a.kv_scale = kv_scale; a.num_pages = num_pages;
    a.ve_h = ve_h; a.ve = ve; a.ve_gate = ve_gate; a.ve_tokens = tokens; a.C = C;
    return launch_append(a, true, stream);
}

}  // namespace nc

using namespace nc;

extern "C" int nc_kv_append_fp8(const void *k, const void *v, long long token_stride, int B, int T, int Hkv,
                                const int32_t *start_pos, const int32_t *num_new, const int32_t *block_table,
                                int max_pages, void *k_pages, void *v_pages, float *kv_scale, int num_pages,
                                void *stream) {
    if (!k || !v || !start_pos || !block_table || !k_pages || !v_pages || !kv_scale) return NC_ERR_NULL;
    if (B <= 0 || T <= 0 || Hkv <= 0 || max_pages <= 0 || num_pages <= 0 || token_stride < (long long)Hkv * HEAD_DIM)
        return NC_ERR_SHAPE;
    if ((long long)B * T > 0x7FFFFFFFLL) return NC_ERR_SHAPE;
    AppendArgs a = {};
    a.k = (const uint16_t *)k;
    a.v = (const uint16_t *)v;
    a.token_stride = token_stride;
    a.B = B; a.T = T; a.Hq = 0; a.Hkv = Hkv;
    a.start_pos = start_pos; a.num_new = num_new;
    a.block_table = block_table; a.max_pages = max_pages;
    a.k_pages = (uint8_t *)k_pages; a.v_pages = (uint8_t *)v_pages;
    a.kv_scale = kv_scale; a.num_pages = num_pages;
    return launch_append(a, false, (hipStream_t)stream);
}

extern "C" int nc_qk_norm_rope_append_fp8(const void *qkv, long long token_stride, int B, int T, int Hq, int Hkv,
                                          const int32_t *start_pos, const int32_t *num_new, const float *q_gain,
                                          const float *k_gain, const float *cos, const float *sin, int rope_len,
                                          void *q_out, const int32_t *block_table, int max_pages, void *k_pages,
                                          void *v_pages, float *kv_scale, int num_pages, void *stream) {
    if (!qkv || !start_pos || !q_gain || !k_gain || !cos || !sin || !q_out || !block_table || !k_pages || !v_pages ||
        !kv_scale)
        return NC_ERR_NULL;
    if (B <= 0 || T <= 0 || Hq <= 0 || Hkv <= 0 || max_pages <= 0 || num_pages <= 0 || rope_len <= 0 ||
        token_stride < (long long)(Hq + 2 * Hkv) * HEAD_DIM)
        return NC_ERR_SHAPE;
    if ((long long)B * T > 0x7FFFFFFFLL) return NC_ERR_SHAPE;
    AppendArgs a = {};
    a.qkv = (const uint16_t *)qkv;
    a.token_stride = token_stride;
    a.B = B; a.T = T; a.Hq = Hq; a.Hkv = Hkv;
    a.start_pos = start_pos; a.num_new = num_new;
    a.q_gain = q_gain; a.k_gain = k_gain; a.cos = cos; a.sin = sin; a.rope_len = rope_len;
    a.q_out = (uint16_t *)q_out;
    a.block_table = block_table; a.max_pages = max_pages;
    a.k_pages = (uint8_t *)k_pages; a.v_pages = (uint8_t *)v_pages;
    a.kv_scale = kv_scale; a.num_pages = num_pages;
    return launch_append(a, true, (hipStream_t)stream);
}

extern "C" int qkp_backward_blocks() { return QKB_BLOCKS; }

extern "C" void qkp_backward(const void *q, const void *k, const void *gq, const void *gk, const void *dqo,
                             const void *dko, void *dq, void *dk, void *dgq, void *dgk, void *part, const void *cos,
                             const void *sin, long long rows, int H, int T, void *stream) {
    if (!q || !k || !gq || !gk || !dqo || !dko || !dq || !dk || !dgq || !dgk || !part || !cos || !sin) {
        last_error = NC_ERR_NULL;
        return;
    }
    if (H <= 0 || T <= 0 || rows < 0 || rows % H) {
        last_error = NC_ERR_SHAPE;
        return;
    }
    hipLaunchKernelGGL(qkp_backward_kernel, dim3(2 * QKB_BLOCKS), dim3(256), 0, (hipStream_t)stream,
                       (const uint16_t *)q, (const uint16_t *)k, (const float *)gq, (const float *)gk,
                       (const uint16_t *)dqo, (const uint16_t *)dko, (uint16_t *)dq, (uint16_t *)dk,
                       (const float *)cos, (const float *)sin, (float *)part, rows / H, H, T);
    hipLaunchKernelGGL(qkp_gain_sum_kernel, dim3(2, HEAD_DIM / 16), dim3(256), 0, (hipStream_t)stream, (const float *)part,
                       (float *)dgq, (float *)dgk);
    last_error = (int)hipGetLastError();
}

extern "C" void qkp_forward(const void *q, const void *k, const void *gq, const void *gk, void *qo, void *ko,
                            const void *cos, const void *sin, long long rows, int H, int T, void *stream) {
    if (!q || !k || !gq || !gk || !qo || !ko || !cos || !sin) {
        last_error = NC_ERR_NULL;
        return;
    }
    if (H <= 0 || T <= 0 || rows <= 0 || rows % H || rows / H > 0x7FFFFFFFLL) {
        last_error = NC_ERR_SHAPE;
        return;
    }
    const dim3 grid((unsigned)((rows / H + 15) / 16 * 2 * qk_head_chunks(H)));
    hipLaunchKernelGGL(qkp_forward_kernel, grid, dim3(256), 0, (hipStream_t)stream, (const uint16_t *)q,
                       (const uint16_t *)k, (const float *)gq, (const float *)gk, (uint16_t *)qo, (uint16_t *)ko,
                       (const float *)cos, (const float *)sin, rows / H, H, T);
    last_error = (int)hipGetLastError();
}

void nc::set_last_error(int status) { last_error = status; }

extern "C" int nc_last_error(void) { return last_error; }

extern "C" const char *nc_status_string(int status) {
    switch (status) {
        case NC_OK: return "ok";
        case NC_ERR_NULL: return "a required pointer is NULL";
        case NC_ERR_SHAPE: return "a size or head count is out of the supported range";
        case NC_ERR_WORKSPACE: return "the workspace is smaller than nc_decode_workspace_bytes";
        default: return status > 0 ? hipGetErrorString((hipError_t)status) : "unknown status";
    }
}

extern "C" int nc_abi_version(void) { return 4; }
