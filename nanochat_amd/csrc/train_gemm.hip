/*
 * The training block's output projection on gfx950: its forward with the residual and the row statistic
 * (linear_residual_rms, on prefill_gemm.hip's tiled kernel) and its weight gradient (weight_grad).
 *
 * weight_grad: out[i][j] += sum_m a[m][i] b[m][j] for token rows m (a = the output's gradient [M][N1], b = the input
 * [M][N2], bf16, fp32 sums). The result is small (C x C) and the sum long (every token), so the tiles alone would leave
 * most of the chip idle (768 x 768: 9 tiles of 256 x 256): the tokens are cut into slices, one workgroup a (tile,
 * slice), each storing its fp32 partial tile, and weight_grad_sum_kernel adds a tile's partials in slice order, so the
 * result does not depend on scheduling. Few tokens, or tiles enough, make one slice, whose tiles are added into the result.
 *
 * Both operands have the summed dimension as their row, so a stage (32 token rows of 256 columns of each operand, 32
 * KiB) goes into LDS as it lies in memory, by LDS DMA, and the MFMA operands are read transposed
 * (ds_read_b64_tr_b16: four rows of one column a lane). A 512-byte LDS row keeps its 32-byte piece s at place
 * s ^ (row % 8), so the eight rows that half a wave reads meet in different banks. Eight waves hold 128 x 64 outputs
 * each; a ring of four stage buffers keeps three in flight, with hand-placed waits and a barrier without a memory fence.
 * 65,536 tokens, 768 x 768: 99 us (783 TFLOP/s) + 13 us for the sum of 28 slices, where the library's GEMM took 297 us on
 * 24 tiles and a pass more to add its result; 9,995 tokens, 1,280 x 1,280: 89 + 6 -> 46 us.
 *
 * linear_residual_rms: 141 us + 5 us for the rows' rstd at 65,536 tokens, C = 768, against a library GEMM with fp32 output
 * (99 us) and five elementwise and reducing passes over it (251 us).
 */
#include "nanochat_amd.h"
#include "nc_device.h"
#include "nc_internal.h"

namespace nc {
namespace {

constexpr int WG_T = 256;                      /* a tile's rows and columns */
constexpr int WG_KC = 32;                      /* tokens per stage */
constexpr int WG_ROWB = WG_T * 2;              /* bytes of a stage's row of one operand */
constexpr int WG_OPB = WG_KC * WG_ROWB;        /* bytes of a stage's operand: 16 KiB */
constexpr int WG_RING = 4;
constexpr int WG_WAVES = 8;
constexpr int WG_LOADS = 2 * WG_OPB / 1024 / WG_WAVES;   /* DMA instructions a wave issues a stage (both operands) */
constexpr int WG_PAST = 0x7FFF0000;            /* a byte offset past every operand's range */

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __amdgpu_buffer_rsrc_t Rsrc;
typedef __attribute__((address_space(3))) void LdsPtr;
typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4i16 LdsV4;

struct WeightGrad {
    const uint16_t *a, *b;     /* [M][N1], [M][N2] bf16 */
    int N1, N2, tiles2;        /* tiles2: column tiles */
    long long M;
    int slices, rows;          /* token slices, rows of each (a multiple of WG_KC) */
    float *part;               /* [slices][N1][N2]; DIRECT: the result [N1][N2], added into */
};

struct WgStage {
    unsigned char a[WG_OPB], b[WG_OPB];
};

/* Stage j's DMA of one operand: rows 32 j .. + 31 of the slice (rows past its end lie outside the range: zeros), columns
 * c0 .. c0 + 255 (past N: no access, zeros). Instruction q moves rows 2 q, 2 q + 1; lane l row 2 q + l / 32, LDS piece
 * (l % 32) / 2, half l % 2. */
__device__ __forceinline__ void wg_fetch(Rsrc rs, unsigned char *lds, int j, int N, int c0, int wave, int lane) {
#pragma unroll
    for (int k = 0; k < WG_LOADS / 2; k++) {
        const int q = wave + WG_WAVES * k, row = 2 * q + (lane >> 5);
        const int piece = ((lane & 31) >> 1) ^ (row & 7), col = c0 + piece * 16 + (lane & 1) * 8;
        const int off = col < N ? ((j * WG_KC + row) * N + col) * 2 : WG_PAST;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (LdsPtr *)(lds + q * 1024), 16, off, 0, 0, 0);
    }
}

/* The MFMA operand of columns 16 d .. + 15 of a stage operand: lane (g, c) gets column 16 d + c of rows 4 g .. + 3, then
 * 16 + 4 g .. + 3. ds_read_b64_tr_b16 hands lane c of a 16-lane group element c % 4 of the 8 bytes lane 4 t + c / 4
 * points at, t = 0 .. 3: lane c points at columns 16 d + 4 (c % 4) .. + 3 of row base + c / 4. */
__device__ __forceinline__ bf16x8 wg_operand(const unsigned char *lds, int d, int g, int c) {
    const int r0 = 4 * g + (c >> 2), r1 = r0 + 16;   /* r0 and r1 share row % 8 */
    const int at = ((d ^ (r0 & 7)) << 5) + ((c & 3) << 3);
    const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsV4 *)(lds + r0 * WG_ROWB + at));
    const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsV4 *)(lds + r1 * WG_ROWB + at));
    const uint2 x = __builtin_bit_cast(uint2, lo), y = __builtin_bit_cast(uint2, hi);
    return __builtin_bit_cast(bf16x8, uint4{x.x, x.y, y.x, y.y});
}

__device__ __forceinline__ void wg_wait_stage() {   /* all but the newest two stages' DMA landed, LDS reads done */
    constexpr int n = (WG_RING - 2) * WG_LOADS;
    __builtin_amdgcn_s_waitcnt((n & 0xF) | ((n >> 4) << 14) | (0x7 << 4) | (0x0 << 8));
}

__device__ __forceinline__ void wg_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

__device__ __forceinline__ void wg_compute(const WgStage &s, f32x4 (&acc)[8][4], int wm, int wn, int g, int c) {
    bf16x8 fb[4];
#pragma unroll
    for (int u = 0; u < 4; u++) fb[u] = wg_operand(s.b, 4 * wn + u, g, c);
#pragma unroll
    for (int t = 0; t < 8; t++) {
        const bf16x8 fa = wg_operand(s.a, 8 * wm + t, g, c);
#pragma unroll
        for (int u = 0; u < 4; u++) acc[t][u] = mfma16x16x32(fa, fb[u], acc[t][u]);
    }
}

/* One ring position: wait for stage j, barrier (every wave's DMA of stage j has landed, every wave is done with stage
 * j - 1), refill stage j - 1's buffer with stage j + 3, compute stage j. */
#define WG_STEP(j, CUR, OLD)                                                          \
    do {                                                                              \
        wg_wait_stage();                                                              \
        wg_barrier();                                                                 \
        wg_fetch(ra, OLD.a, (j) + WG_RING - 1, p.N1, i0, wave, lane);                 \
        wg_fetch(rb, OLD.b, (j) + WG_RING - 1, p.N2, j0, wave, lane);                 \
        wg_compute(CUR, acc, wm, wn, g, c);                                           \
    } while (0)

/* DIRECT: one slice, whose tiles are added straight into the result. */
template <bool DIRECT>
__global__ void __launch_bounds__(WG_WAVES *WAVE, 1) weight_grad_kernel(WeightGrad p) {
    __shared__ __align__(16) WgStage s0, s1, s2, s3;   /* distinct objects: a read of one never waits for another's DMA */
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
    const int wm = wave >> 2, wn = wave & 3;
    /* slices fastest: the workgroups that run together read different tokens of the same few columns */
    const int slice = blockIdx.x % p.slices, tile = blockIdx.x / p.slices;
    const int i0 = tile / p.tiles2 * WG_T, j0 = tile % p.tiles2 * WG_T;
    const long long m0 = (long long)slice * p.rows;
    const int rows = (int)(p.M - m0 < p.rows ? p.M - m0 : p.rows);   /* > 0: the host makes no empty slice */
    const Rsrc ra = __builtin_amdgcn_make_buffer_rsrc((void *)(p.a + m0 * p.N1), (short)0, rows * p.N1 * 2, 0x00020000);
    const Rsrc rb = __builtin_amdgcn_make_buffer_rsrc((void *)(p.b + m0 * p.N2), (short)0, rows * p.N2 * 2, 0x00020000);
    const int stages = (rows + WG_KC - 1) / WG_KC;
    f32x4 acc[8][4];
#pragma unroll
    for (int t = 0; t < 8; t++)
#pragma unroll
        for (int u = 0; u < 4; u++) acc[t][u] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    wg_fetch(ra, s0.a, 0, p.N1, i0, wave, lane);
    wg_fetch(rb, s0.b, 0, p.N2, j0, wave, lane);
    wg_fetch(ra, s1.a, 1, p.N1, i0, wave, lane);
    wg_fetch(rb, s1.b, 1, p.N2, j0, wave, lane);
    wg_fetch(ra, s2.a, 2, p.N1, i0, wave, lane);
    wg_fetch(rb, s2.b, 2, p.N2, j0, wave, lane);
    for (int j = 0; j < stages; j += WG_RING) {   /* stages past the slice read zeros and add nothing */
        WG_STEP(j, s0, s3);
        WG_STEP(j + 1, s1, s0);
        WG_STEP(j + 2, s2, s1);
        WG_STEP(j + 3, s3, s2);
    }
    __builtin_amdgcn_s_waitcnt(0);   /* no DMA may land in LDS after the workgroup ends */
    /* lane (g, c) of result tile (t, u): rows i0 + 128 wm + 16 t + 4 g + e, column j0 + 64 wn + 16 u + c. 32-bit offsets into
     * the tile's rows (flat addresses took 2 us more at 2,048 tokens, and spilled where the tile is added): rows past N1 lie
     * outside them, columns past N2 take an offset past them, and neither is accessed. */
    const int live = p.N1 - i0 < WG_T ? p.N1 - i0 : WG_T;
    const unsigned row_bytes = (unsigned)p.N2 * 4;
    const Rsrc ro = __builtin_amdgcn_make_buffer_rsrc((void *)(p.part + ((long long)slice * p.N1 + i0) * p.N2), (short)0,
                                                      live * (int)row_bytes, 0x00020000);
    unsigned at[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const int col = j0 + 64 * wn + 16 * u + c;
        at[u] = col < p.N2 ? (unsigned)(128 * wm + 4 * g) * row_bytes + (unsigned)col * 4 : (unsigned)WG_PAST;
    }
    float old[2][4][4];   /* DIRECT: the result's rows of t, and of t + 1 in flight (one tile at a time waited 32 times) */
    const auto fetch_old = [&](int t) {
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int e = 0; e < 4; e++)
                old[t & 1][u][e] =
                    __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(ro, at[u] + (16 * t + e) * row_bytes, 0, 0));
    };
    if (DIRECT) fetch_old(0);
#pragma unroll
    for (int t = 0; t < 8; t++) {
        if (DIRECT && t < 7) fetch_old(t + 1);
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int e = 0; e < 4; e++)
                __builtin_amdgcn_raw_buffer_store_b32(
                    __float_as_uint(DIRECT ? old[t & 1][u][e] + acc[t][u][e] : acc[t][u][e]), ro,
                    at[u] + (16 * t + e) * row_bytes, 0, 0);
    }
}

/* out += the slices' partials added in order; four elements a thread. */
__global__ void __launch_bounds__(256) weight_grad_sum_kernel(const float4 *part, int slices, long long n4, float4 *out) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n4) return;
    float4 sum = part[i];
#pragma unroll 8
    for (int s = 1; s < slices; s++) {
        const float4 v = part[s * n4 + i];
        sum.x = sum.x + v.x; sum.y = sum.y + v.y; sum.z = sum.z + v.z; sum.w = sum.w + v.w;
    }
    const float4 o = out[i];
    out[i] = float4{o.x + sum.x, o.y + sum.y, o.z + sum.z, o.w + sum.w};
}

constexpr int WG_MIN_ROWS = 4 * WG_KC;   /* a shorter slice is mostly the ring's start */

/* What M tokens of an N1 x N2 result take in us by a model of three measured parts, one workgroup (128 KiB of LDS) a CU:
 * - rounds of workgroups, each as long as a slice's stages and ten more for its start and its end;
 * - a stage: 0.65 alone, 20 % more with every CU at work, and then up to 27 % more where the slices, five or more and no
 *   multiple of four, spread over the eight XCDs (workgroup b runs on XCD b % 8 and takes slice b % slices), so that each L2
 *   holds most of them: 1,664 x 1,664 over 65,536 tokens, 49 tiles: 4 slices 341 us, 5 slices 429;
 * - a slice's partial tiles out and back, and the sum; one slice has neither (its tiles are added into the result). */
double weight_grad_time(long long tiles, long long elements, int cus, long long slices, long long rows) {
    const double rounds = (double)((tiles * slices + cus - 1) / cus), busy = (double)(tiles * slices) / (rounds * cus);
    const double spread = slices < 5 || slices % 4 == 0 ? 0.0 : slices % 2 == 0 ? 0.15 : 0.27;
    const double stage = 0.65 * (1.0 + 0.2 * busy + spread * busy * busy);
    const double partials = slices == 1 ? 0.0 : 2.0 + slices * (elements * 1.2e-6 + 0.04);
    return rounds * (rows / WG_KC + 10) * stage + partials;
}

/* Token slices: the best of a few counts by weight_grad_time (small ones, steps of about a quarter above, and those that just
 * fill one to four rounds), none under WG_MIN_ROWS rows unless it is the only one and none whose operand slice passes 1
 * GiB. As many as fill the CUs, and one where the tiles are half of them or more, left CUs idle at wide results and spent
 * more on partials than they saved at few tokens. us, so and by the model (library product and addition):
 *   tokens    768 x 768        1,664 x 1,664      2,560 x 2,560       3,072 x 3,072
 *      512    17 -> 15 (25)      23 ->  21 (25)     34 ->  23 (31)      37 ->    26 (41)
 *    2,048    24 -> 22 (27)      37 ->  31 (32)     47 ->  47 (51)      64 ->    53 (67)
 *    9,995    36 -> 29 (66)      85 ->  69 (104)   122 -> 122 (157)    212 ->   190 (214)
 *   65,536    80 -> 80 (298)    429 -> 341 (605)   752 -> 742 (1,075) 1,411 -> 1,044 (1,159)
 * Over 64 .. 65,536 tokens and 1 .. 289 tiles its pick is within 1 % of the best of these counts on average. */
void weight_grad_slices(long long M, int N1, int N2, int &slices, int &rows) {
    const long long tiles = (long long)((N1 + WG_T - 1) / WG_T) * ((N2 + WG_T - 1) / WG_T);
    const long long fit = (1LL << 30) / ((N1 > N2 ? N1 : N2) * 2) / WG_KC * WG_KC;
    const long long least = (M + fit - 1) / fit, most = (M + WG_MIN_ROWS - 1) / WG_MIN_ROWS;
    const int cus = device_cus();
    double best = -1.0;
    slices = rows = 0;
    auto consider = [&](long long s) {
        s = s < most ? s : most;
        s = s > least ? s : least;
        const long long r = ((M + s - 1) / s + WG_KC - 1) / WG_KC * WG_KC;
        if (r > fit) return;
        s = (M + r - 1) / r;   /* no empty slice */
        const double t = weight_grad_time(tiles, (long long)N1 * N2, cus, s, r);
        if (best >= 0.0 && t >= best) return;
        best = t;
        slices = (int)s;
        rows = (int)r;
    };
    for (long long s = 1; s <= most && (s == 1 || tiles * s <= 4LL * cus); s += s < 8 ? 1 : s / 4) consider(s);
    for (int k = 1; k <= 4; k++)
        if (k * cus >= tiles) consider(k * cus / tiles);
}

/* One slice needs none (never 0 where there is a call). */
long long weight_grad_bytes(int slices, int N1, int N2) { return slices == 1 ? 16 : (long long)slices * N1 * N2 * 4; }

bool weight_grad_fits(long long M, int N1, int N2) {
    return M >= 0 && M < (1LL << 40) && N1 > 0 && N2 > 0 && N1 % 8 == 0 && N2 % 8 == 0 && N1 <= 65536 && N2 <= 65536;
}

}  // namespace
}  // namespace nc

using namespace nc;

extern "C" long long nc_weight_grad_workspace_bytes(long long rows, int n1, int n2) {
    if (!weight_grad_fits(rows, n1, n2)) return -1;
    if (rows == 0) return 0;
    int slices, per;
    weight_grad_slices(rows, n1, n2, slices, per);
    return weight_grad_bytes(slices, n1, n2);
}

extern "C" int nc_weight_grad(const void *a, const void *b, long long rows, int n1, int n2, float *out, void *workspace,
                              long long workspace_bytes, void *stream) {
    if (!weight_grad_fits(rows, n1, n2)) return NC_ERR_SHAPE;
    if (rows == 0) return NC_OK;
    if (!a || !b || !out || !workspace) return NC_ERR_NULL;
    if (((uintptr_t)a | (uintptr_t)b | (uintptr_t)out | (uintptr_t)workspace) & 15) return NC_ERR_SHAPE;
    WeightGrad p;
    p.a = (const uint16_t *)a; p.b = (const uint16_t *)b;
    p.N1 = n1; p.N2 = n2; p.tiles2 = (n2 + WG_T - 1) / WG_T;
    p.M = rows;
    weight_grad_slices(rows, n1, n2, p.slices, p.rows);
    if (workspace_bytes < weight_grad_bytes(p.slices, n1, n2)) return NC_ERR_WORKSPACE;
    p.part = (float *)workspace;
    const long long tiles = (long long)((n1 + WG_T - 1) / WG_T) * p.tiles2;
    const dim3 grid((unsigned)(tiles * p.slices)), block(WG_WAVES * WAVE);
    if (p.slices == 1) {
        p.part = out;
        hipLaunchKernelGGL(weight_grad_kernel<true>, grid, block, 0, (hipStream_t)stream, p);
        return (int)hipGetLastError();
    }
    hipLaunchKernelGGL(weight_grad_kernel<false>, grid, block, 0, (hipStream_t)stream, p);
    const long long n4 = (long long)n1 * n2 / 4;
    hipLaunchKernelGGL(weight_grad_sum_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       (const float4 *)workspace, p.slices, n4, (float4 *)out);
    return (int)hipGetLastError();
}

/* Row chunks under prefill_gemm's 2 GiB arrays (fp32 sized), a multiple of its 256-row tiles. */
static long long lrr_chunk(int n, int k) { return ((1LL << 31) - 1) / (4LL * (n > k ? n : k)) / 256 * 256; }

extern "C" int nc_linear_residual_rms(const void *x, const void *w, const void *res, long long rows, int n, int k,
                                      void *out, float *rstd, void *workspace, long long workspace_bytes,
                                      void *stream) {
    if (rows < 0 || n <= 0 || k <= 0 || k % 128 || n % 4 || (long long)n * k * 2 >= (1LL << 31) || n > 65536 ||
        k > 65536 || rows > (1LL << 40))
        return NC_ERR_SHAPE;
    if (rows == 0) return NC_OK;
    if (!x || !w || !res || !out || !rstd || !workspace) return NC_ERR_NULL;
    if (((uintptr_t)x | (uintptr_t)w) & 15 || ((uintptr_t)res | (uintptr_t)out) & 7 || ((uintptr_t)workspace & 3))
        return NC_ERR_SHAPE;
    if (workspace_bytes < rows * pf_ssq_cols(n) * 4) return NC_ERR_WORKSPACE;
    const long long chunk = lrr_chunk(n, k);
    float *ssq = (float *)workspace;
    for (long long m = 0; m < rows; m += chunk) {
        const int mm = (int)(rows - m < chunk ? rows - m : chunk);
        PfGemm g = {(const uint16_t *)x + m * k, (const uint16_t *)w, mm, n, k, (uint16_t *)out + m * n, nullptr,
                    (const uint16_t *)res + m * n, nullptr, ssq + m * pf_ssq_cols(n)};
        const int e = prefill_gemm(g, SG_RESID2, (hipStream_t)stream);
        if (e != 0) return e;
        const int e2 = tile_rstd(g.ssq, mm, n, rstd + m, (hipStream_t)stream);
        if (e2 != 0) return e2;
    }
    return NC_OK;
}
