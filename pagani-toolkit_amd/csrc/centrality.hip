// centrality.hip -- eigenvector centrality and participation coefficient,
// MI355X (gfx950).
//
//  * Eigenvector centrality (U/CUEC/CUEC/CUEC_unweighted.cu:61-196, W/CUEC/
//    weighted-net.cu:55-203): the reference's power iteration -- start vector
//    0..n-1; per iteration u0 = u, |u|, u *= 1/|u|, u = A u, err1 = |u - u0|,
//    err2 = |u + u0|; stop when either is <= 1e-6 or after 10000 iterations --
//    as one launch per iteration.  Rows are split over a fixed set of blocks;
//    every block first reduces the previous launch's per-block partials (|u|^2,
//    |u - u0|^2, |u + u0|^2) in a fixed order, so all blocks take the same stop
//    decision on the device and launches past the stop return at once.  The
//    host looks once per batch of launches.  FP64 throughout, FP32 weights.
//    The SpMV stages segments of the vector in LDS, or, for a sparse network,
//    gathers it (pg_spmv.hpp).
//  * Participation coefficient (W/PC_CPU/PC_CPU/main.cpp:96-160): one wave per
//    vertex, FP32 module sums accumulated in LDS in CSR order by one lane
//    (entries staged 64 at a time), then the FP32 sum of squared shares over
//    modules 1..K in order -- the reference's arithmetic, so bit-identical.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "pg_internal.hpp"
#include "pg_spmv.hpp"

namespace {

constexpr int EC_MAX_ITER = 10000;  // CUEC_unweighted.cu:25
constexpr double EC_EPS = 1e-6;     // CUEC_unweighted.cu:28
constexpr int EC_TPB = pgdev::SP_TPB;
constexpr int EC_BATCH = 32;        // launches per host check

// rows of block b
struct EcBlock {
    int n, R;
    __device__ __forceinline__ void operator()(int b, int &a0, int &nr) const
    {
        a0 = b * R;
        nr = min(n - a0, R);
    }
};

struct EcState {
    int stopped, iters;  // stopped: 1 + the launch that found the stop, 0 before
    double lam, err1, err2;
};

// Block b owns rows [b R, b R + R); partials |u - u_prev|^2, |u + u_prev|^2, |u|^2.
__global__ __launch_bounds__(EC_TPB) void ec_init(int n, int R, double *__restrict__ u, double *__restrict__ part,
                                                  EcState *__restrict__ st)
{
    __shared__ double red[EC_TPB / 64 * 3];
    const int i0 = blockIdx.x * R, nr = min(n - i0, R);
    double s[3] = {0.0, 0.0, 0.0};
    if ((int)threadIdx.x < nr) {
        const double x = (double)(i0 + (int)threadIdx.x);
        u[i0 + threadIdx.x] = x;
        s[2] = x * x;
    }
    pgdev::sp_block_sums<3>(s, nr, red, part + 3 * blockIdx.x);
    if (blockIdx.x == 0 && threadIdx.x == 0) *st = EcState{0, 0, 0.0, 1.0, 1.0};
}

// Iteration k.  Every block takes the norm and the stop decision from the
// previous launch's partials, then its rows of A u by the SpMV of
// pg_spmv.hpp on the raw u, scaled once per row.  Staged, n = 40,009 with 16 M entries:
// 20.0 us (27.1 us with one lane per row in blocks of 256 rows; 21.9 us with a
// segment's first entries loaded behind its staging), three segments of about
// 5 us each, bound by the entries' latency from beyond L2 (32 MB of them an
// iteration), not by the look-ups: leaving out the fillers' changed nothing.
template <bool W, bool GATHER>
__global__ __launch_bounds__(EC_TPB) void ec_iter(const int *__restrict__ row, pgdev::SpLayout L, int n, int R, int G, int k,
                                                  const double *__restrict__ uin, double *__restrict__ uout,
                                                  double *__restrict__ vhat, const double *__restrict__ pin,
                                                  double *__restrict__ pout, EcState *__restrict__ st)
{
    extern __shared__ double xs[];
    __shared__ double rowv[pgdev::SP_ROWS];
    __shared__ int2 pt[pgdev::SP_ROWS];
    __shared__ double red[EC_TPB / 64 * 3], tot[3];
    // only a stop of an earlier launch counts: block 0 of this one may set it
    // while other blocks start, and the waves of a block have to agree (all
    // reach that same decision from the partials)
    const int stop = st->stopped;
    if (stop > 0 && stop <= k) return;
    const int tid = threadIdx.x;
    const int i0 = blockIdx.x * R, nr = min(n - i0, R);
    const int im = tid < nr ? i0 + (int)L.perm[i0 + tid] : n - 1;  // slot tid's row
    double ui, t;
    bool empty;
    const bool go = pgdev::sp_product<W, GATHER>(L, i0, nr, uin, n, xs, pt, rowv, [&]() {
        ui = uin[im];
        empty = row[im] == row[im + 1];
        double a[3];
        pgdev::sp_partials<3>(pin, 0, G, a, tot);
        if (k > 0) {
            const double e1 = sqrt(a[0]), e2 = sqrt(a[1]);
            if (!(e1 > EC_EPS && e2 > EC_EPS) || k >= EC_MAX_ITER) {
                if (blockIdx.x == 0 && tid == 0) {
                    st->err1 = e1;
                    st->err2 = e2;
                    st->iters = k;
                    st->stopped = k + 1;
                }
                return false;
            }
        }
        const double vnorm = sqrt(a[2]);
        t = 1 / vnorm;
        if (blockIdx.x == 0 && tid == 0) st->lam = vnorm;
        return true;
    });
    if (!go) return;
    double s[3] = {0.0, 0.0, 0.0};
    if (tid < nr) {
        const int i = im;
        const double y = empty ? 0.0 : rowv[tid] * t;  // t = inf once u = 0
        vhat[i] = ui * t;
        uout[i] = y;
        const double d1 = y - ui, d2 = y + ui;
        s[0] = d1 * d1;
        s[1] = d2 * d2;
        s[2] = y * y;
    }
    pgdev::sp_block_sums<3>(s, nr, red, pout + 3 * blockIdx.x);
}

// ------------------------------------------------ participation coefficient

// flags[0] |= label < 1; flags[1] = max label
__global__ void label_scan(const int *__restrict__ lab, int n, int *__restrict__ flags)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int l = lab[i];
    if (l < 1) atomicOr(&flags[0], 1);
    atomicMax(&flags[1], l);
}

__global__ __launch_bounds__(64) void pc_kernel(const int *__restrict__ row, const int *__restrict__ col,
                                                const float *__restrict__ val, const int *__restrict__ lab, int n,
                                                int K, float *__restrict__ pc, float *__restrict__ pcn)
{
#pragma clang fp contract(off)
    extern __shared__ float wm[];  // K module sums
    __shared__ int sm_m[64];
    __shared__ float sm_v[64];
    const int i = blockIdx.x, lane = threadIdx.x;
    const int a = row[i], b = row[i + 1];
    for (int j = lane; j < K; j += 64) wm[j] = 0.0f;
    float deg = 0.0f;  // lane 0: the reference's sequential FP32 sum
    for (int base = a; base < b; base += 64) {
        const int e = base + lane;
        if (e < b) {
            sm_m[lane] = lab[col[e]] - 1;
            sm_v[lane] = val ? val[e] : 1.0f;
        }
        __syncthreads();
        if (lane == 0) {
            const int cnt = min(64, b - base);
            for (int q = 0; q < cnt; q++) {
                deg += sm_v[q];
                wm[sm_m[q]] += sm_v[q];
            }
        }
        __syncthreads();
    }
    if (lane != 0) return;
    float r;
    if (deg == 0) {
        r = 0.0f;
    } else {
        float sum = 0.0f;
        for (int j = 0; j < K; j++) {
            const float t = wm[j] / deg;
            sum += t * t;
        }
        r = 1.0f - sum;
    }
    pc[i] = r;
    if (pcn) pcn[i] = K != 1 ? r / ((float)(K - 1) / (float)K) : r;
}

}  // namespace

extern "C" pg_status pg_eigenvector_centrality(pg_ctx *ctx, const int32_t *row, const int32_t *col,
                                               const float *val, int32_t n, int64_t nnz, double *vhat,
                                               double *avec, double *lambda, int32_t *iters)
{
    if (!ctx) return PG_EINVAL;
    PG_HIP(ctx, hipSetDevice(ctx->device));
    PG_TRY(pg_check_csr_args(ctx, row, col, n, nnz));
    if (n < 1) return pg_fail(ctx, PG_EINVAL, "n must be >= 1");
    const int *drow, *dcol;
    const float *dval = nullptr;
    PG_TRY(pg_in(ctx, row, (size_t)n + 1, "in.row", &drow));
    PG_TRY(pg_in(ctx, col, (size_t)nnz, "in.col", &dcol));
    if (val) PG_TRY(pg_in(ctx, val, (size_t)nnz, "in.val", &dval));
    PG_TRY(pg_validate_csr(ctx, drow, dcol, n, nnz, true));
    hipStream_t st = ctx->stream;
    // about one block per CU (its LDS holds a vector segment)
    const int R = (int)std::min<long long>(pgdev::SP_ROWS, std::max<long long>(16, pg_cdiv(n, std::max(ctx->num_cu, 1))));
    const int G = (int)pg_cdiv(n, R);
    pgdev::SpLayout L{};
    const bool gather = pgdev::sp_gathers(n, nnz, G);
    int *parts;
    if (gather) {
        PG_TRY(pg_bufT(ctx, "ec.gcol", (size_t)nnz, &L.gcol));
        if (dval) PG_TRY(pg_bufT(ctx, "ec.val", (size_t)nnz, &L.val));
        PG_TRY(pg_bufT(ctx, "ec.part", 2 * (size_t)n, &parts));
    } else {
        L.nseg = pgdev::sp_nseg(n);
        L.cap = pgdev::sp_cap(n);
        const size_t room = pgdev::sp_room(n, nnz, L.nseg);
        PG_TRY(pg_bufT(ctx, "ec.idx", room, &L.idx));
        if (dval) PG_TRY(pg_bufT(ctx, "ec.val", room, &L.val));
        PG_TRY(pg_bufT(ctx, "ec.part", 2 * (size_t)n * L.nseg, &parts));
    }
    const size_t lds = gather ? 0 : pgdev::sp_lds(L.cap);
    const auto iter_fn = gather ? (dval ? ec_iter<true, true> : ec_iter<false, true>)
                                : (dval ? ec_iter<true, false> : ec_iter<false, false>);
    if (!gather)
        PG_HIP(ctx, hipFuncSetAttribute((const void *)iter_fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    PG_TRY(pg_bufT(ctx, "ec.perm", (size_t)n, &L.perm));
    L.part = (int2 *)parts;
    pgdev::sp_build<<<(unsigned)pg_cdiv(n, 4), 256, 0, st>>>(drow, dcol, dval, n, nullptr, nullptr, 0, nullptr, nullptr,
                                                            L, nullptr, 0);
    pgdev::sp_order<<<(unsigned)G, pgdev::SP_TPB, 0, st>>>(drow, (const int *)nullptr, EcBlock{n, R}, L.perm);
    PG_KERNEL_CHECK(ctx);
    double *u[2], *part[2], *dvh, *dav;
    EcState *dst;
    PG_TRY(pg_bufT(ctx, "ec.u0", (size_t)n, &u[0]));
    PG_TRY(pg_bufT(ctx, "ec.u1", (size_t)n, &u[1]));
    PG_TRY(pg_bufT(ctx, "ec.p0", 3 * (size_t)G, &part[0]));
    PG_TRY(pg_bufT(ctx, "ec.p1", 3 * (size_t)G, &part[1]));
    PG_TRY(pg_bufT(ctx, "ec.state", 1, &dst));
    PG_TRY(pg_out(ctx, vhat, (size_t)n, "out.ecvhat", &dvh));
    if (!dvh) PG_TRY(pg_bufT(ctx, "ec.vhat", (size_t)n, &dvh));
    // iteration k reads u[k & 1] and part[(k + 1) & 1], writes the other two;
    // ec_init fills u[0] and part[1]
    ec_init<<<(unsigned)G, EC_TPB, 0, st>>>(n, R, u[0], part[1], dst);
    PG_KERNEL_CHECK(ctx);
    EcState h{};
    for (int k0 = 0; k0 <= EC_MAX_ITER; k0 += EC_BATCH) {
        for (int k = k0; k < k0 + EC_BATCH && k <= EC_MAX_ITER; k++)
            iter_fn<<<(unsigned)G, EC_TPB, lds, st>>>(drow, L, n, R, G, k, u[k & 1], u[(k + 1) & 1], dvh,
                                                      part[(k + 1) & 1], part[k & 1], dst);
        PG_KERNEL_CHECK(ctx);
        PG_HIP(ctx, hipMemcpyAsync(&h, dst, sizeof h, hipMemcpyDeviceToHost, st));
        PG_HIP(ctx, hipStreamSynchronize(st));
        if (h.stopped) break;
    }
    if (!h.stopped) return pg_fail(ctx, PG_EDEVICE, "power iteration did not stop");
    // the last executed iteration (iters - 1) wrote y into u[iters & 1]
    PG_TRY(pg_out_finish(ctx, vhat, dvh, (size_t)n));
    if (avec) {
        PG_TRY(pg_out(ctx, avec, (size_t)n, "out.ecavec", &dav));
        PG_HIP(ctx, hipMemcpyAsync(dav, u[h.iters & 1], (size_t)n * 8, hipMemcpyDeviceToDevice, st));
        PG_TRY(pg_out_finish(ctx, avec, dav, (size_t)n));
    }
    PG_HIP(ctx, hipStreamSynchronize(st));
    if (lambda) *lambda = h.lam;
    if (iters) *iters = h.iters;
    return PG_OK;
}

extern "C" pg_status pg_participation(pg_ctx *ctx, const int32_t *row, const int32_t *col, const float *val,
                                      int32_t n, int64_t nnz, const int32_t *labels, float *pc,
                                      float *pc_norm, int32_t *nmod)
{
    if (!ctx) return PG_EINVAL;
    PG_HIP(ctx, hipSetDevice(ctx->device));
    PG_TRY(pg_check_csr_args(ctx, row, col, n, nnz));
    if (n < 1 || !labels || !pc) return pg_fail(ctx, PG_EINVAL, "bad arguments");
    const int *drow, *dcol, *dlab;
    const float *dval = nullptr;
    PG_TRY(pg_in(ctx, row, (size_t)n + 1, "in.row", &drow));
    PG_TRY(pg_in(ctx, col, (size_t)nnz, "in.col", &dcol));
    if (val) PG_TRY(pg_in(ctx, val, (size_t)nnz, "in.val", &dval));
    PG_TRY(pg_in(ctx, labels, (size_t)n, "in.labels", &dlab));
    PG_TRY(pg_validate_csr(ctx, drow, dcol, n, nnz, false));
    hipStream_t st = ctx->stream;
    int *flags, hf[2] = {0, 0};
    PG_TRY(pg_bufT(ctx, "pc.flags", 2, &flags));
    PG_HIP(ctx, hipMemsetAsync(flags, 0, 8, st));
    label_scan<<<(unsigned)pg_cdiv(n, 256), 256, 0, st>>>(dlab, n, flags);
    PG_KERNEL_CHECK(ctx);
    PG_HIP(ctx, hipMemcpyAsync(hf, flags, 8, hipMemcpyDeviceToHost, st));
    PG_HIP(ctx, hipStreamSynchronize(st));
    if (hf[0]) return pg_fail(ctx, PG_EINVAL, "module labels must be >= 1");
    const int K = hf[1];
    const size_t lds = (size_t)K * sizeof(float);
    if (lds > ctx->lds_per_block - 1024)
        return pg_fail(ctx, PG_ENOTSUP, "%d modules exceed the LDS budget of one wave", K);
    float *dpc, *dpn;
    PG_TRY(pg_out(ctx, pc, (size_t)n, "out.pc", &dpc));
    PG_TRY(pg_out(ctx, pc_norm, (size_t)n, "out.pcn", &dpn));
    pc_kernel<<<(unsigned)n, 64, lds, st>>>(drow, dcol, dval, dlab, n, K, dpc, dpn);
    PG_KERNEL_CHECK(ctx);
    PG_TRY(pg_out_finish(ctx, pc, dpc, (size_t)n));
    PG_TRY(pg_out_finish(ctx, pc_norm, dpn, (size_t)n));
    PG_HIP(ctx, hipStreamSynchronize(st));
    if (nmod) *nmod = K;
    return PG_OK;
}
