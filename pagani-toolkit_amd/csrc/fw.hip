// fw.hip -- blocked Floyd-Warshall APSP on MI355X (gfx950) VALUs.
//
// Replaces cuAPSP (W/Lp/CUBFW_Lp/CUBFW_Lp/CUBFW.cpp:19-168) and the phase
// kernels of CUBFW_ph1.cu / CUBFW_ph2.cu / CUBFW_ph3.cu.  The whole padded
// matrix stays resident in HBM (the reference streams every tile over PCIe each
// round).  Per k-block round:
//   phase 1: the diagonal tile, sequential k over register micro-tiles (one
//            work-group; from the second round on inside phase 3 of the round
//            before);
//   phase 2: row and column panel tiles, sequential k, 16 lanes per column or row;
//   phase 3: every other tile, min over k of (ik + kj), 4x4 register
//            micro-tiles over LDS panels.
// Min-plus is not a dense contraction, so this runs on VALU (v_add_f32 +
// v_min3_f32), not MFMA.  Each candidate path length is one FP32 add of the
// same operands as the blocked CPU algorithm (W/Lp/CUBFW_Lp/CUBFW_Lp/BFW.cpp:
// 40-108) with the same tile edge, and min is exact, so the result is
// bit-identical to it.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "pg_internal.hpp"

namespace {

__device__ __forceinline__ float relax(float cur, float cand) { return cand < cur ? cand : cur; }

// The tile edge's micro-tiles: 4 x 4 per thread, (B/4)^2 threads: 256 for B =
// 64, 1024 for B = 128.
template <int B>
constexpr int fw_threads() { return (B / 4) * (B / 4); }

// Sequential closure of a diagonal tile held in registers: at step k the
// threads holding row k and column k publish them to a double-buffered LDS row
// / column (one barrier per step), everyone relaxes its micro-tile against
// them.  Row and column k do not change during step k (d_kk = 0), as in the
// sequential reference loop, so every element sees the same operands there.
template <int B>
__device__ __forceinline__ void fw_closure(float (&acc)[4][4], int tx, int ty, float (*rowk)[B], float (*colk)[B])
{
    constexpr int M = 4;
    for (int q = 0; q < B / M; q++) {  // k = q M + kk
#pragma unroll
        for (int kk = 0; kk < M; kk++) {
            const int buf = kk & 1;
            if (ty == q)
#pragma unroll
                for (int b = 0; b < M; b++) rowk[buf][tx * M + b] = acc[kk][b];
            if (tx == q)
#pragma unroll
                for (int a = 0; a < M; a++) colk[buf][ty * M + a] = acc[a][kk];
            __syncthreads();
            float ik[M], kj[M];
#pragma unroll
            for (int a = 0; a < M; a++) ik[a] = colk[buf][ty * M + a];
#pragma unroll
            for (int b = 0; b < M; b++) kj[b] = rowk[buf][tx * M + b];
#pragma unroll
            for (int a = 0; a < M; a++)
#pragma unroll
                for (int b = 0; b < M; b++) acc[a][b] = relax(acc[a][b], ik[a] + kj[b]);
        }
    }
}

template <int B>
__device__ __forceinline__ void fw_tile_load(const float *__restrict__ d, int np, long long r, long long c, float (&acc)[4][4])
{
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
        for (int b = 0; b < 4; b++) acc[a][b] = d[(r + a) * np + c + b];
}

template <int B>
__device__ __forceinline__ void fw_tile_store(float *__restrict__ d, int np, long long r, long long c, const float (&acc)[4][4])
{
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
        for (int b = 0; b < 4; b++) d[(r + a) * np + c + b] = acc[a][b];
}

// Phase 1 of the first round (later rounds' run inside phase 3).
template <int B>
__global__ __launch_bounds__(fw_threads<B>()) void fw_diag(float *__restrict__ d, int np)
{
    __shared__ float rowk[2][B], colk[2][B];
    constexpr int TS = B / 4;
    const int tx = threadIdx.x % TS, ty = threadIdx.x / TS;
    float acc[4][4];
    fw_tile_load<B>(d, np, ty * 4, tx * 4, acc);
    fw_closure<B>(acc, tx, ty, rowk, colk);
    fw_tile_store<B>(d, np, ty * 4, tx * 4, acc);
}

// x of lane Q of the caller's row of 16 lanes (DPP row_newbcast).
template <int Q>
__device__ __forceinline__ float row_bcast(float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x150 + Q, 0xf, 0xf, true));
}

// One panel lane's steps k = Q M .. B - 1: v[r] = min(v[r], g[k][r] + v_k), v_k
// the row's value k from lane k / M, g the closed diagonal (LDS).
template <int B, int Q>
__device__ __forceinline__ void fw_panel_steps(float (&v)[B / 16], const float (*g)[B + 4], int at)
{
    constexpr int M = B / 16;
#pragma unroll
    for (int kk = 0; kk < M; kk++) {
        const float vk = row_bcast<Q>(v[kk]);
#pragma unroll
        for (int r = 0; r < M; r++) v[r] = relax(v[r], g[Q * M + kk][at + r] + vk);
    }
    if constexpr (Q + 1 < 16) fw_panel_steps<B, Q + 1>(v, g, at);
}

// Phase 2.  In a row panel every column is on its own (d_ij = min(d_ij, diag_ik
// + d_kj), k in order), in a column panel every row (d_ij = min(d_ij, d_ik +
// diag_kj)).  Each takes 16 lanes, M = B / 16 values a lane; value k reaches
// the others by a DPP broadcast within the 16 lanes, so the B sequential steps
// need no barrier and no LDS round trip in their chain.  Work-groups of 16
// columns or rows: B / 16 per tile, row panels first.  B = 64: 10.9 us a round
// at n = 4,160 (25 us with the tile shared by a work-group and a barrier per
// step).
template <int B>
__global__ __launch_bounds__(256) void fw_panels(float *__restrict__ d, int np, int kb)
{
    constexpr int M = B / 16, PER = B / 16;
    __shared__ __align__(16) float g[B][B + 4];  // row panels: diag transposed, g[k][i]; column panels: g[k][j]
    const int h = (np / B - 1) * PER;
    const bool rows = (int)blockIdx.x < h;  // row panel
    const int x = rows ? blockIdx.x : blockIdx.x - h;
    int t = x / PER;
    t = t < kb ? t : t + 1;
    const long long k0 = (long long)kb * B, p0 = (long long)t * B + (x % PER) * 16;  // first column (row) of the 16
    const int tid = threadIdx.x, one = tid >> 4, at = (tid & 15) * M;
    float v[M];
#pragma unroll
    for (int r = 0; r < M; r++)
        v[r] = rows ? d[(k0 + at + r) * np + p0 + one] : d[(p0 + one) * np + k0 + at + r];
    float w[B * B / 256];
#pragma unroll
    for (int u = 0; u < B * B / 256; u++) w[u] = d[(k0 + (tid + u * 256) / B) * np + k0 + (tid + u * 256) % B];
#pragma unroll
    for (int u = 0; u < B * B / 256; u++) {
        const int i = (tid + u * 256) / B, j = (tid + u * 256) % B;
        if (rows) g[j][i] = w[u];
        else g[i][j] = w[u];
    }
    __syncthreads();
    fw_panel_steps<B, 0>(v, g, at);
#pragma unroll
    for (int r = 0; r < M; r++) {
        if (rows) d[(k0 + at + r) * np + p0 + one] = v[r];
        else d[(p0 + one) * np + k0 + at + r] = v[r];
    }
}

// Phase 3: tile (r, c) = min(tile, min_k ik[i][k] + kj[k][j]) for r, c != kb.
// The work-group of the next round's diagonal tile goes on to close it: that
// tile is final here, its 64 dependent steps pass under the other tiles, and
// the next round starts with its panels.  It is block (0, 0), so it starts
// first.  (B = 128: 134 KB of LDS panels allow one work-group per CU.)
template <int B>
__global__ __launch_bounds__(fw_threads<B>()) void fw_phase3(float *__restrict__ d, int np, int kb)
{
    constexpr int M = 4;
    constexpr int TS = B / M;           // threads per tile edge
    constexpr int NT = fw_threads<B>();
    __shared__ float sa[B][B + 1];  // ik panel, [i][k]
    __shared__ float sb[B][B + 4];  // kj panel, [k][j]
    const int nbk = np / B;
    int r = blockIdx.y, c = blockIdx.x;
    const bool next = kb + 1 < nbk;
    bool diag = false;
    if (next) {  // places (0, 0) and (kb, kb), the next diagonal's, trade
        if (r == 0 && c == 0) {
            r = c = kb;
            diag = true;
        } else if (r == kb && c == kb) {
            r = c = 0;
        }
    }
    r = r < kb ? r : r + 1;
    c = c < kb ? c : c + 1;
    if (r >= nbk || c >= nbk) return;
    const int tid = threadIdx.x, tx = tid % TS, ty = tid / TS;
    const long long r0 = (long long)r * B, c0 = (long long)c * B, k0 = (long long)kb * B;
    for (int e = tid; e < B * B; e += NT) {
        int i = e / B, j = e % B;
        sa[i][j] = d[(r0 + i) * np + k0 + j];
        sb[i][j] = d[(k0 + i) * np + c0 + j];
    }
    float acc[M][M];
    fw_tile_load<B>(d, np, r0 + ty * M, c0 + tx * M, acc);
    __syncthreads();
    for (int k = 0; k < B; k += 2) {
        float x0[M], x1[M], y0[M], y1[M];
#pragma unroll
        for (int a = 0; a < M; a++) {
            x0[a] = sa[ty * M + a][k];
            x1[a] = sa[ty * M + a][k + 1];
        }
#pragma unroll
        for (int b = 0; b < M; b++) {
            y0[b] = sb[k][tx * M + b];
            y1[b] = sb[k + 1][tx * M + b];
        }
#pragma unroll
        for (int a = 0; a < M; a++)
#pragma unroll
            for (int b = 0; b < M; b++) acc[a][b] = fminf(acc[a][b], fminf(x0[a] + y0[b], x1[a] + y1[b]));
    }
    if (diag) {
        __syncthreads();  // the panels' LDS is free
        fw_closure<B>(acc, tx, ty, (float(*)[B])&sa[0][0], (float(*)[B])&sb[0][0]);
    }
    fw_tile_store<B>(d, np, r0 + ty * M, c0 + tx * M, acc);
}

__global__ void fw_pad_in(const float *__restrict__ src, int n, float *__restrict__ dst, int np)
{
    long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= (long long)np * np) return;
    long long i = k / np, j = k % np;
    dst[k] = (i < n && j < n) ? src[i * n + j] : (i == j ? 0.0f : INFINITY);
}

__global__ void fw_pad_out(const float *__restrict__ src, int np, float *__restrict__ dst, int n)
{
    long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= (long long)n * n) return;
    long long i = k / n, j = k % n;
    dst[k] = src[i * np + j];
}

// W FormBlock.cpp:52-74 in row-major: edge distances, then 0 on the diagonal.
// One work-group per row fills and scatters it (a thread per row took 198 us at
// n = 4,099, after 23 us of filling).  A row whose columns do not ascend
// strictly may repeat one, and the last entry wins: one thread scatters it.
__global__ __launch_bounds__(256) void fw_from_csr(const int *__restrict__ row, const int *__restrict__ col,
                                                   const float *__restrict__ val, int n, int kind, float *__restrict__ d)
{
    const int i = blockIdx.x;
    float *di = d + (long long)i * n;
    for (int j = threadIdx.x; j < n; j += 256) di[j] = j == i ? 0.0f : INFINITY;
    const int a = row[i], b = row[i + 1];
    bool unsorted = false;
    for (int e = a + (int)threadIdx.x; e + 1 < b; e += 256) unsorted = unsorted || col[e] >= col[e + 1];
    unsorted = __syncthreads_or(unsorted) != 0;  // and the fill is done
    for (int e = a + (unsorted ? 0 : (int)threadIdx.x); e < b && (!unsorted || threadIdx.x == 0); e += unsorted ? 1 : 256) {
        const int j = col[e];
        if (j == i) continue;
        const float w = val ? val[e] : 1.0f;
        di[j] = kind == 0 ? 1.0f / w : (kind == 1 ? 1.0f - w : 1.0f);
    }
}

// One block per row u: e_u and the FP64 row sum for Lp (CUBFW_Lp.cpp:70-113).
__global__ __launch_bounds__(256) void fw_eff_rows(const float *__restrict__ d, int n, float *__restrict__ eff,
                                                  double *__restrict__ rowsum, int *__restrict__ iso)
{
    __shared__ float rf[256];
    __shared__ double rd[256];
    const int u = blockIdx.x, tid = threadIdx.x;
    float sf = 0.0f;
    double sd = 0.0;
    for (int v = tid; v < n; v += 256) {
        const float x = d[(long long)u * n + v];
        if (v == u || !(x >= 0.1f)) continue;  // the reference skips d < 0.1
        const float q = 1.0f / x;
        sf += q;
        sd += (double)q;
    }
    rf[tid] = sf;
    rd[tid] = sd;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (tid < o) {
            rf[tid] += rf[tid + o];
            rd[tid] += rd[tid + o];
        }
        __syncthreads();
    }
    if (tid == 0) {
        float e = n > 1 ? rf[0] / (float)(n - 1) : 0.0f;
        if (e < 1.0f / (float)n) {
            e = 0.0f;
            atomicAdd(iso, 1);
        }
        if (eff) eff[u] = e;
        rowsum[u] = rd[0];
    }
}

__global__ __launch_bounds__(256) void fw_lp_sum(const double *__restrict__ rowsum, int n, double *__restrict__ out)
{
    __shared__ double r[256];
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) s += rowsum[i];
    r[threadIdx.x] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) r[threadIdx.x] += r[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = r[0];
}

template <int B>
pg_status fw_run(pg_ctx *ctx, float *dm, int np)
{
    hipStream_t st = ctx->stream;
    const int nbk = np / B;
    fw_diag<B><<<1, fw_threads<B>(), 0, st>>>(dm, np);
    for (int kb = 0; kb < nbk && nbk > 1; kb++) {
        fw_panels<B><<<2 * (nbk - 1) * (B / 16), 256, 0, st>>>(dm, np, kb);
        fw_phase3<B><<<dim3(nbk - 1, nbk - 1), fw_threads<B>(), 0, st>>>(dm, np, kb);
    }
    PG_KERNEL_CHECK(ctx);
    return PG_OK;
}

}  // namespace

extern "C" pg_status pg_fw(pg_ctx *ctx, float *d, int32_t n, int32_t block)
{
    if (!ctx) return PG_EINVAL;
    if (!d || n < 0) return pg_fail(ctx, PG_EINVAL, "bad arguments");
    if (block == 0 && n > 0 && pg_autotune_on_first_use(ctx) && pg_tune_get(ctx, "fw_block", n, 0, 0) == 0) {
        pg_tune_result tr;
        PG_TRY(pg_autotune_fw(ctx, d, n, &tr));
    }
    if (block == 0) {
        // a value forced by the autotuner's search, else the tuned one for
        // (arch, n), else 64 (measured faster than 128 at N = 8192)
        block = ctx->force_fw_block;
        if (block <= 0) block = pg_tune_get(ctx, "fw_block", n, 0, 0);
        if (block != 64 && block != 128) block = 64;
    }
    if (block != 64 && block != 128) return pg_fail(ctx, PG_EINVAL, "tile edge %d: use 64 or 128", block);
    if (n == 0) return PG_OK;
    PG_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t st = ctx->stream;
    const int np = (int)pg_cdiv(n, block) * block;
    const long long nn = (long long)n * n, npp = (long long)np * np;
    const bool dev = pg_is_device_ptr(d);
    float *dm = nullptr;
    float *din = d;
    if (!dev) {
        PG_TRY(pg_bufT(ctx, "fw.in", (size_t)nn, &din));
        PG_HIP(ctx, hipMemcpyAsync(din, d, nn * 4, hipMemcpyHostToDevice, st));
    }
    if (np == n) {
        dm = din;
    } else {
        PG_TRY(pg_bufT(ctx, "fw.pad", (size_t)npp, &dm));
        fw_pad_in<<<(unsigned)pg_cdiv(npp, 256), 256, 0, st>>>(din, n, dm, np);
    }
    if (block == 64) PG_TRY(fw_run<64>(ctx, dm, np));
    else PG_TRY(fw_run<128>(ctx, dm, np));
    if (np != n) fw_pad_out<<<(unsigned)pg_cdiv(nn, 256), 256, 0, st>>>(dm, np, din, n);
    PG_KERNEL_CHECK(ctx);
    if (!dev) PG_HIP(ctx, hipMemcpyAsync(d, din, nn * 4, hipMemcpyDeviceToHost, st));
    PG_HIP(ctx, hipStreamSynchronize(st));
    return PG_OK;
}

extern "C" pg_status pg_fw_init(pg_ctx *ctx, const int32_t *row, const int32_t *col, const float *val,
                                int32_t n, int64_t nnz, int32_t kind, float *d)
{
    if (!ctx) return PG_EINVAL;
    if (!d || kind < 0 || kind > 2 || (kind != 2 && !val)) return pg_fail(ctx, PG_EINVAL, "bad arguments");
    PG_TRY(pg_check_csr_args(ctx, row, col, n, nnz));
    PG_HIP(ctx, hipSetDevice(ctx->device));
    const int *drow, *dcol;
    const float *dval = nullptr;
    PG_TRY(pg_in(ctx, row, (size_t)n + 1, "in.row", &drow));
    PG_TRY(pg_in(ctx, col, (size_t)nnz, "in.col", &dcol));
    if (val) PG_TRY(pg_in(ctx, val, (size_t)nnz, "in.val", &dval));
    PG_TRY(pg_validate_csr(ctx, drow, dcol, n, nnz, false));
    const long long nn = (long long)n * n;
    float *dd;
    PG_TRY(pg_out(ctx, d, (size_t)nn, "out.fw", &dd));
    hipStream_t st = ctx->stream;
    if (nn > 0) fw_from_csr<<<(unsigned)n, 256, 0, st>>>(drow, dcol, dval, n, kind, dd);
    PG_KERNEL_CHECK(ctx);
    PG_TRY(pg_out_finish(ctx, d, dd, (size_t)nn));
    PG_HIP(ctx, hipStreamSynchronize(st));
    return PG_OK;
}

extern "C" pg_status pg_fw_efficiency(pg_ctx *ctx, const float *d, int32_t n, float *eff, double *lp,
                                      int32_t *isolated)
{
    if (!ctx) return PG_EINVAL;
    if (!d || n < 1) return pg_fail(ctx, PG_EINVAL, "bad arguments");
    PG_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t st = ctx->stream;
    const float *dd;
    PG_TRY(pg_in(ctx, d, (size_t)n * n, "fw.in", &dd));
    float *de;
    double *rs, *tot;
    int *iso;
    PG_TRY(pg_out(ctx, eff, (size_t)n, "out.eff", &de));
    PG_TRY(pg_bufT(ctx, "fw.rowsum", (size_t)n, &rs));
    PG_TRY(pg_bufT(ctx, "fw.lpsum", 1, &tot));
    PG_TRY(pg_bufT(ctx, "fw.iso", 1, &iso));
    PG_HIP(ctx, hipMemsetAsync(iso, 0, 4, st));
    fw_eff_rows<<<(unsigned)n, 256, 0, st>>>(dd, n, de, rs, iso);
    fw_lp_sum<<<1, 256, 0, st>>>(rs, n, tot);
    PG_KERNEL_CHECK(ctx);
    PG_TRY(pg_out_finish(ctx, eff, de, (size_t)n));
    double s = 0.0;
    int ni = 0;
    PG_HIP(ctx, hipMemcpyAsync(&s, tot, 8, hipMemcpyDeviceToHost, st));
    PG_HIP(ctx, hipMemcpyAsync(&ni, iso, 4, hipMemcpyDeviceToHost, st));
    PG_HIP(ctx, hipStreamSynchronize(st));
    if (lp) {
        double x = s;
        x /= n;
        x /= (n - 1);
        *lp = 1.0 / x;
    }
    if (isolated) *isolated = ni;
    return PG_OK;
}
