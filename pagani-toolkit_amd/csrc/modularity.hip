// modularity.hip -- Newman leading-eigenvector modularity on MI355X (gfx950).
//
// Replaces Partition_GPU / Sub_Partition_GPU / Lead_Vector_GPU
// (W/Newman_Modularity_GPU/CUmodularity/modularity_GPU.cu:225-525) and the CPU
// twins used for groups of up to 25000 nodes (Modularity_CPU.cpp:164-298).
// The power iteration on B^(g) + beta I is one CSR SpMV (FP32 weights, FP64
// accumulation) plus the rank-one degree term and the diagonal correction; all
// norms and dot products are FP64 on the device.  Every round whose members
// are known (a wave) iterates together: one launch per iteration covers all
// of the wave's groups, each group stops on the device at the reference's
// test, and the host checks the wave once per BATCH iterations.
//
// The bisection bookkeeping (group membership, label order) is host code like
// the reference's Partition_GPU and runs in the reference's round order, so
// labels match it; the groups' edges are laid out on the device.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "pg_internal.hpp"
#include "pg_spmv.hpp"

namespace {

constexpr int MAX_ITER = 10000;      // modularity_GPU.cu:25
constexpr double EPS = 1e-6;         // modularity_GPU.cu:28
constexpr double RAYLEIGH_TOL = 1e-8;  // default relative tolerance of the quotient stop
constexpr int TPB = pgdev::SP_TPB;   // threads per block
constexpr int NPB_MAX = pgdev::SP_ROWS;  // nodes per work block, upper limit
constexpr int GSUM_MAX = 512;        // target for block partials per group
constexpr int BATCH = 64;            // power iterations queued per host check

// A work block's group and the group's ranges, one scalar load.
struct Block {
    int g, fb, nb, no, ng, pad[3];
};

// nodes of work block b
struct ModBlock {
    const Block *blk;
    int npb;
    __device__ __forceinline__ void operator()(int b, int &a0, int &nr) const
    {
        const Block B = blk[b];
        a0 = B.no + (b - B.fb) * npb;
        nr = min(B.no + B.ng - a0, npb);
    }
};

// One wave of independent groups (the rounds created but not yet processed),
// concatenated: group g owns nodes [no[g], no[g] + ng[g]) of the wave and
// blocks [fb[g], fb[g] + nb[g]); a block never spans two groups, so every
// per-group sum is a fixed-order sum of its blocks' partials.
struct Wave {
    int nnodes, nblk;
    int npb;               // nodes per work block (16 .. NPB_MAX)
    const Block *blk;      // [nblk]
    const int *no, *ng, *fb, *nb;   // [G]
    const int *gid;        // [nnodes] global id (start vector)
    pgdev::SpLayout lay;   // edges inside the groups, columns relative to the group
    const double *k, *sumbg;
    double m2;
    int stopmode;          // pg_mod_stop
    double tol;            // Rayleigh-quotient tolerance
    int max_iter;          // iterations per pass
    // per group state
    int ngroups;
    int *iters;
    int2 *state;           // [G] stopped, launch index the pass began with
    const int *restart;    // [G] 1: (re)start the group's pass from the start vector
    double *beta, *lam;
    // vectors: y_li, the result of iteration li before normalising (li = 0:
    // the start vector, not normalised), is in buf[li % 3]; its norm (1 for
    // li = 0) in vn[3 g + li % 3]
    double *buf[3], *vn, *vres;
    // per-block partials of the launch with the iteration's parity
    double *part[2];
    double *rho;           // [G][2] Rayleigh quotient of iteration li in rho[2 g + (li & 1)]
};

// |y|^2, y . k, and by the stopping rule v . y and v . v, or |v - v_prev|^2
// and |v + v_prev|^2
enum { P_YY, P_YK, P_A, P_B, NPART };

// Iteration li of a group (li = launches since its pass began) is one launch:
// from the previous launch's partials come the norm of y_li, v_li . k and the
// quotient of iteration li - 1 (the Rayleigh stop); then
//   y_(li+1) = (B^(g) + beta I) v_li,  v_li = y_li / |y_li|,
// a CSR SpMV of the raw y_li (pg_spmv.hpp; FP32 weights, FP64 sums) scaled once
// per row, with the partials of |y|^2, y . k, v . y, v . v.  |v_li -+ v_(li-1)|
// needs |y_li|, so its partials are taken here too and the vector stop looks
// at them one launch later: the launch that finds it leaves y_li and y_(li-1)
// in place.  n = 14,011 with 4.9 M weighted entries: 9.3 us an iteration, half of
// it the launch and the chain of loads up to the first row (55 us as two
// launches that gathered the vector from L2 with a wave per row, four per
// CU).  Every skip below is uniform in a block.
template <bool W, bool GATHER>
__global__ __launch_bounds__(TPB) void mod_iter(Wave w, int it)
{
    extern __shared__ double xs[];
    __shared__ double rowv[NPB_MAX];
    __shared__ int2 pt[NPB_MAX];
    __shared__ double red[TPB / 64 * NPART], tot[NPART];
    __shared__ int skip;
    const int tid = threadIdx.x, b = blockIdx.x;
    const Block B = w.blk[b];
    const int2 state = w.state[B.g];
    const int li = it - state.y;  // iterations completed in this pass
    const double *y = w.buf[li % 3], *yp = w.buf[(li + 2) % 3];
    double *yn = w.buf[(li + 1) % 3];
    const int i0 = B.no + (b - B.fb) * w.npb, nr = min(B.no + B.ng - i0, w.npb);
    const bool vec = w.stopmode == PG_MOD_STOP_VECTOR;
    const int i = tid < nr ? i0 + (int)w.lay.perm[i0 + tid] : i0;  // slot tid's node
    double yi, ki, si, ypi, beta, vnp, vn, sum[NPART];
    const bool go = pgdev::sp_product<W, GATHER>(w.lay, i0, nr, y + B.no, B.ng, xs, pt, rowv, [&]() {
        // every load that does not wait for the partials goes out before them
        yi = y[i];
        ki = w.k[i];
        si = w.sumbg[i];
        ypi = vec ? yp[i] : 0.0;
        beta = w.beta[B.g];
        vnp = w.vn[3 * B.g + (li + 2) % 3];
        // the stop flag may be set by this launch's first block of the group;
        // every block of it reaches the same decision below, so either
        // reading skips
        if (tid == 0) skip = state.x;
        pgdev::sp_partials<NPART>(w.part[(it + 1) & 1], B.fb, B.nb, sum, tot);  // its barrier publishes skip
        if (skip) return false;
        const bool lead = b == B.fb && tid == 0;
        vn = li > 0 ? sqrt(sum[P_YY]) : 1.0;
        if (lead) w.vn[3 * B.g + li % 3] = vn;
        if (li == 0) return true;
        int done = 0, at = li;
        if (vec) {
            if (li > 1) {
                const double e1 = sqrt(sum[P_A]), e2 = sqrt(sum[P_B]);
                done = !(e1 > EPS && e2 > EPS);
                if (done) at = li - 1;
            }
        } else {
            // quotients of the last two completed iterations
            const double ra = sum[P_A] / sum[P_B];
            if (lead) w.rho[2 * B.g + ((li - 1) & 1)] = ra;
            if (li >= 2) {
                const double rb = w.rho[2 * B.g + (li & 1)];
                done = fabs(ra - rb) <= w.tol * fabs(ra);
            }
        }
        if (!done && li < w.max_iter) return true;
        if (lead) {
            w.iters[B.g] = at;
            w.state[B.g].x = 1;
        }
        return false;
    });
    if (!go) return;
    const double sc = 1.0 / vn, vk = sum[P_YK] * sc;
    double p[NPART] = {0.0, 0.0, 0.0, 0.0};
    if (tid < nr) {
        const double x = yi * sc;
        const double acc = rowv[tid] * sc - (vk / w.m2 * ki + (si - beta) * x);
        yn[i] = acc;
        p[P_YY] = acc * acc;
        p[P_YK] = acc * ki;
        if (!vec) {
            p[P_A] = x * acc;
            p[P_B] = x * x;
        } else if (li > 0) {
            const double xp = ypi / vnp;
            p[P_A] = (x - xp) * (x - xp);
            p[P_B] = (x + xp) * (x + xp);
        }
    }
    pgdev::sp_block_sums<NPART>(p, nr, red, w.part[it & 1] + (long long)b * NPART);
}

// Groups flagged in restart[]: buf[0] = global ids (the start vector) and the
// partials of x . k, as left by the launch before the pass's first, it.
__global__ __launch_bounds__(TPB) void mod_start(Wave w, int it)
{
    __shared__ double red[TPB / 64 * NPART];
    const int b = blockIdx.x;
    const Block B = w.blk[b];
    if (!w.restart[B.g]) return;
    const int i0 = B.no + (b - B.fb) * w.npb, nr = min(B.no + B.ng - i0, w.npb);
    double p[NPART] = {0.0, 0.0, 0.0, 0.0};
    if ((int)threadIdx.x < nr) {
        const int i = i0 + threadIdx.x;
        const double x = (double)w.gid[i];
        w.buf[0][i] = x;
        p[P_YK] = x * w.k[i];
    }
    pgdev::sp_block_sums<NPART>(p, nr, red, w.part[(it + 1) & 1] + (long long)b * NPART);
}

// For the groups in list[]: lam[g] = +-|y| by the sign of v[mi] v0[mi] at the
// first largest |v[mi]| (the reference's strict '>' scan), v = the final
// vector, v0 = the one before (Rayleigh stop: the last quotient); vres[] = v.
__global__ __launch_bounds__(TPB) void mod_lambda(Wave w, const int *list)
{
    __shared__ double rv[TPB];
    __shared__ int ri[TPB];
    const int g = list[blockIdx.x], tid = threadIdx.x;
    const int a = w.no[g], z = a + w.ng[g];
    const int li = w.iters[g];
    const double *y = w.buf[li % 3], *y0 = w.buf[(li + 2) % 3];
    const double vn = w.vn[3 * g + li % 3], vn0 = w.vn[3 * g + (li + 2) % 3];
    double best = -1.0;
    int bi = 0x7fffffff;
    for (int i = a + tid; i < z; i += TPB) {
        const double v = y[i] / vn, x = fabs(v);
        w.vres[i] = v;
        if (x > best) { best = x; bi = i; }
    }
    rv[tid] = best;
    ri[tid] = bi;
    __syncthreads();
    for (int o = TPB / 2; o > 0; o >>= 1) {
        if (tid < o) {
            const double x = rv[tid + o];
            const int ix = ri[tid + o];
            if (x > rv[tid] || (x == rv[tid] && ix < ri[tid])) { rv[tid] = x; ri[tid] = ix; }
        }
        __syncthreads();
    }
    if (tid == 0) {
        const int mi = ri[0];
        if (w.stopmode == PG_MOD_STOP_RAYLEIGH) w.lam[g] = w.rho[2 * g + ((li - 1) & 1)];
        else w.lam[g] = (mi < z && (y[mi] / vn) * (y0[mi] / vn0) > 0) ? vn : -vn;
    }
}

// k of every vertex: degree, or the FP64 sum of its weights (one wave per row).
__global__ __launch_bounds__(256) void mod_strength(const int *__restrict__ row, const float *__restrict__ val, int n,
                                                    double *__restrict__ k)
{
    const int i = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (i >= n) return;
    const int a = row[i], b = row[i + 1];
    double s = 0.0;
    if (val) {
        for (int e = a + lane; e < b; e += 64) s += (double)val[e];
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    } else {
        s = (double)(b - a);
    }
    if (lane == 0) k[i] = s;
}

// sumbg[a] = kin[a] - k_i K_g / 2m, i = gid[a]; kw[a] = k_i.  In place of kin.
__global__ void mod_correction(const int *__restrict__ gid, const int *__restrict__ res, int r0,
                               const double *__restrict__ k, const double *__restrict__ Kg, double m2, int nnodes,
                               double *__restrict__ kw, double *__restrict__ sumbg)
{
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= nnodes) return;
    const int i = gid[a];
    kw[a] = k[i];
    sumbg[a] = sumbg[a] - k[i] * Kg[res[i] - r0] / m2;
}

// Per row the FP64 weight (count without val) of its entries inside its own module.
__global__ __launch_bounds__(256) void mod_inside(const int *__restrict__ row, const int *__restrict__ col,
                                                  const float *__restrict__ val, const int *__restrict__ lab, int n,
                                                  double *__restrict__ in)
{
    const int i = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (i >= n) return;
    const int l = lab[i];
    double s = 0.0;
    for (int e = row[i] + lane; e < row[i + 1]; e += 64)
        if (lab[col[e]] == l) s += val ? (double)val[e] : 1.0;
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (lane == 0) in[i] = s;
}

}  // namespace

extern "C" pg_status pg_modularity(pg_ctx *ctx, const int32_t *row, const int32_t *col, const float *val,
                                   int32_t n, int64_t nnz, int32_t kmode, int32_t *labels, double *q,
                                   double *lambda0, double *eig0, int32_t *rounds)
{
    pg_mod_opts o;
    std::memset(&o, 0, sizeof o);
    o.kmode = kmode;
    o.stop = PG_MOD_STOP_VECTOR;
    return pg_modularity_ex(ctx, row, col, val, n, nnz, &o, labels, q, lambda0, eig0, rounds);
}

extern "C" pg_status pg_modularity_ex(pg_ctx *ctx, const int32_t *row, const int32_t *col, const float *val,
                                      int32_t n, int64_t nnz, const pg_mod_opts *opts, int32_t *labels,
                                      double *q, double *lambda0, double *eig0, int32_t *rounds)
{
    if (!ctx) return PG_EINVAL;
    if (!labels || !opts) return pg_fail(ctx, PG_EINVAL, "labels/opts is NULL");
    const int kmode = opts->kmode;
    if (kmode != PG_MOD_STRENGTH && kmode != PG_MOD_BINARY_K) return pg_fail(ctx, PG_EINVAL, "bad kmode");
    if (opts->stop != PG_MOD_STOP_VECTOR && opts->stop != PG_MOD_STOP_RAYLEIGH)
        return pg_fail(ctx, PG_EINVAL, "bad stop rule %d", opts->stop);
    if (opts->tol < 0.0 || opts->max_iter < 0 || opts->max_depth < 0)
        return pg_fail(ctx, PG_EINVAL, "bad tol / max_iter / max_depth");
    const double tol = opts->tol > 0.0 ? opts->tol : RAYLEIGH_TOL;
    const int max_iter = opts->max_iter > 0 ? opts->max_iter : MAX_ITER;
    PG_TRY(pg_check_csr_args(ctx, row, col, n, nnz));
    PG_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t st = ctx->stream;
    const int *drow, *dcol;
    const float *dval = nullptr;
    PG_TRY(pg_in(ctx, row, (size_t)n + 1, "in.row", &drow));
    PG_TRY(pg_in(ctx, col, (size_t)nnz, "in.col", &dcol));
    if (val) PG_TRY(pg_in(ctx, val, (size_t)nnz, "in.val", &dval));
    PG_TRY(pg_validate_csr(ctx, drow, dcol, n, nnz, false));
    const size_t nn = (size_t)n + 1;
    double *d_kall, *d_in;
    int *d_res, *d_rloc, *d_part;
    PG_TRY(pg_bufT(ctx, "mod.kall", nn, &d_kall));
    PG_TRY(pg_bufT(ctx, "mod.inside", nn, &d_in));
    PG_TRY(pg_bufT(ctx, "mod.res", nn, &d_res));
    PG_TRY(pg_bufT(ctx, "mod.rloc", nn, &d_rloc));
    // edges inside the groups of a wave: sized, and their form chosen, once for
    // the whole network
    const int npb0 = (int)std::min<long long>(NPB_MAX, std::max<long long>(16, pg_cdiv(n, std::max(ctx->num_cu, 1))));
    const bool gather = pgdev::sp_gathers(n, nnz, pg_cdiv(n, npb0));
    pgdev::SpLayout lay{};
    {
        const int nseg = gather ? 1 : pgdev::sp_nseg(n);
        const size_t room = gather ? (size_t)nnz : pgdev::sp_room(n, nnz, nseg);
        if (gather) PG_TRY(pg_bufT(ctx, "mod.gcol", room, &lay.gcol));
        else PG_TRY(pg_bufT(ctx, "mod.idx", room, &lay.idx));
        if (dval) PG_TRY(pg_bufT(ctx, "mod.lval", room, &lay.val));
        PG_TRY(pg_bufT(ctx, "mod.part", 2 * nn * nseg, &d_part));
        lay.part = (int2 *)d_part;
        PG_TRY(pg_bufT(ctx, "mod.perm", nn, &lay.perm));
    }

    std::vector<double> k((size_t)n);
    double m2 = 0.0;
    if (n > 0) {
        mod_strength<<<(unsigned)pg_cdiv(n, 4), 256, 0, st>>>(drow, kmode == PG_MOD_BINARY_K ? nullptr : dval, n, d_kall);
        PG_KERNEL_CHECK(ctx);
        PG_HIP(ctx, hipMemcpyAsync(k.data(), d_kall, (size_t)n * 8, hipMemcpyDeviceToHost, st));
        PG_HIP(ctx, hipStreamSynchronize(st));
    }
    for (int i = 0; i < n; i++) m2 += k[i];
    std::vector<int> res((size_t)n, 0), adj((size_t)2 * n + 2, 0);
    int maxr = 0, index = 1, nrounds = 0;
    if (lambda0) *lambda0 = 0.0;
    if (n == 0 || m2 <= 0.0) {
        for (int i = 0; i < n; i++) res[i] = 0;
        adj[0] = 1;
        maxr = -1;
    }

    // Rounds are processed in waves: every round created by the previous wave
    // has fixed membership, so the whole wave's power iterations run together;
    // the bookkeeping (splits, new round numbers, labels) then runs in round
    // order exactly as the sequential driver (modularity_GPU.cu:405-525).
    int lo = 0, nwave = 0;
    std::vector<int> rloc((size_t)n);
    // PAGANI_MOD_TRACE=1: one line per wave on stderr (groups, nodes,
    // iterations, seconds)
    const char *trace_env = std::getenv("PAGANI_MOD_TRACE");
    const bool trace = opts->progress || (trace_env && trace_env[0] == '1');
    while (lo <= maxr) {
        const int hi = maxr + 1;
        const int G = hi - lo;
        if (opts->max_depth > 0 && nwave >= opts->max_depth) {
            // depth limit: this level's groups are final, labelled in round order
            std::vector<char> used((size_t)G, 0);
            for (int i = 0; i < n; i++)
                if (res[i] >= lo && res[i] < hi) used[res[i] - lo] = 1;
            for (int g = 0; g < G; g++)
                if (used[g]) adj[lo + g] = index++;
            break;
        }
        const auto wave_t0 = std::chrono::steady_clock::now();
        // members of each round, in increasing global id
        std::vector<int> gcount((size_t)G, 0);
        for (int i = 0; i < n; i++)
            if (res[i] >= lo && res[i] < hi) gcount[res[i] - lo]++;
        std::vector<int> no((size_t)G), ng((size_t)G), fb((size_t)G), nb((size_t)G);
        int nnodes = 0, nblk = 0;
        // about one work block per CU (its LDS holds a vector segment), none
        // over two groups, no group with more than GSUM_MAX block partials
        int gmax = 1;
        long long all = 0;
        for (int g = 0; g < G; g++) {
            gmax = std::max(gmax, gcount[g]);
            all += gcount[g];
        }
        int npb = (int)std::min<long long>(NPB_MAX, std::max<long long>(16, pg_cdiv(all, std::max(ctx->num_cu, 1))));
        while (npb < NPB_MAX && pg_cdiv(gmax, npb) > GSUM_MAX) npb = std::min(NPB_MAX, 2 * npb);
        for (int g = 0; g < G; g++) {
            no[g] = nnodes;
            ng[g] = gcount[g];
            fb[g] = nblk;
            nb[g] = (int)std::max<long long>(1, pg_cdiv(ng[g], npb));
            nnodes += ng[g];
            nblk += nb[g];
        }
        std::vector<int> gid((size_t)nnodes), fill(no);
        std::vector<Block> blk((size_t)nblk);
        for (int g = 0; g < G; g++)
            for (int q = 0; q < nb[g]; q++) blk[fb[g] + q] = Block{g, fb[g], nb[g], no[g], ng[g], {0, 0, 0}};
        for (int i = 0; i < n; i++)
            if (res[i] >= lo && res[i] < hi) {
                const int g = res[i] - lo;
                rloc[i] = fill[g];
                gid[fill[g]++] = i;
            }
        std::vector<double> Kg((size_t)G, 0.0);
        for (int a = 0; a < nnodes; a++) Kg[res[gid[a]] - lo] += k[gid[a]];

        Wave w;
        Block *d_blk;
        int2 *d_state;
        int *d_no, *d_ng, *d_fb, *d_nb, *d_gid, *d_restart, *d_iters, *d_list;
        double *d_k, *d_sumbg, *d_Kg, *d_beta, *d_lam, *d_vn, *d_vres, *d_rho;
        PG_TRY(pg_bufT(ctx, "mod.blk", (size_t)nblk, &d_blk));
        PG_TRY(pg_bufT(ctx, "mod.no", (size_t)G, &d_no));
        PG_TRY(pg_bufT(ctx, "mod.ng", (size_t)G, &d_ng));
        PG_TRY(pg_bufT(ctx, "mod.fb", (size_t)G, &d_fb));
        PG_TRY(pg_bufT(ctx, "mod.nb", (size_t)G, &d_nb));
        PG_TRY(pg_bufT(ctx, "mod.gid", (size_t)nnodes + 1, &d_gid));
        PG_TRY(pg_bufT(ctx, "mod.k", (size_t)nnodes + 1, &d_k));
        PG_TRY(pg_bufT(ctx, "mod.sumbg", (size_t)nnodes + 1, &d_sumbg));
        PG_TRY(pg_bufT(ctx, "mod.Kg", (size_t)G, &d_Kg));
        PG_TRY(pg_bufT(ctx, "mod.restart", (size_t)G, &d_restart));
        PG_TRY(pg_bufT(ctx, "mod.state", (size_t)G, &d_state));
        PG_TRY(pg_bufT(ctx, "mod.iters", (size_t)G, &d_iters));
        PG_TRY(pg_bufT(ctx, "mod.list", (size_t)G, &d_list));
        PG_TRY(pg_bufT(ctx, "mod.beta", (size_t)G, &d_beta));
        PG_TRY(pg_bufT(ctx, "mod.lam", (size_t)G, &d_lam));
        PG_TRY(pg_bufT(ctx, "mod.vn", (size_t)G * 3, &d_vn));
        PG_TRY(pg_bufT(ctx, "mod.b0", (size_t)nnodes + 1, &w.buf[0]));
        PG_TRY(pg_bufT(ctx, "mod.b1", (size_t)nnodes + 1, &w.buf[1]));
        PG_TRY(pg_bufT(ctx, "mod.b2", (size_t)nnodes + 1, &w.buf[2]));
        PG_TRY(pg_bufT(ctx, "mod.vres", (size_t)nnodes + 1, &d_vres));
        PG_TRY(pg_bufT(ctx, "mod.part0", (size_t)nblk * NPART, &w.part[0]));
        PG_TRY(pg_bufT(ctx, "mod.part1", (size_t)nblk * NPART, &w.part[1]));
        PG_TRY(pg_bufT(ctx, "mod.rho", (size_t)G * 2, &d_rho));
        auto h2d = [&](void *dst, const void *src, size_t bytes) -> pg_status {
            if (bytes) PG_HIP(ctx, hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, st));
            return PG_OK;
        };
        std::vector<int2> hstate((size_t)G, make_int2(0, 0));
        std::vector<double> dzeros((size_t)G, 0.0);
        PG_TRY(h2d(d_blk, blk.data(), (size_t)nblk * sizeof(Block)));
        PG_TRY(h2d(d_no, no.data(), (size_t)G * 4));
        PG_TRY(h2d(d_ng, ng.data(), (size_t)G * 4));
        PG_TRY(h2d(d_fb, fb.data(), (size_t)G * 4));
        PG_TRY(h2d(d_nb, nb.data(), (size_t)G * 4));
        PG_TRY(h2d(d_gid, gid.data(), (size_t)nnodes * 4));
        PG_TRY(h2d(d_Kg, Kg.data(), (size_t)G * 8));
        PG_TRY(h2d(d_res, res.data(), (size_t)n * 4));
        PG_TRY(h2d(d_rloc, rloc.data(), (size_t)n * 4));
        // the groups' edges, laid out on the device
        lay.nseg = gather ? 0 : pgdev::sp_nseg(gmax);
        lay.cap = gather ? 0 : pgdev::sp_cap(gmax);
        pgdev::sp_build<<<(unsigned)pg_cdiv(std::max(nnodes, 1), 4), 256, 0, st>>>(
            drow, dcol, dval, nnodes, d_gid, d_res, lo, d_no, d_rloc, lay, d_sumbg, kmode == PG_MOD_BINARY_K ? 1 : 0);
        pgdev::sp_order<<<(unsigned)nblk, pgdev::SP_TPB, 0, st>>>(drow, (const int *)d_gid, ModBlock{d_blk, npb}, lay.perm);
        mod_correction<<<(unsigned)pg_cdiv(std::max(nnodes, 1), 256), 256, 0, st>>>(d_gid, d_res, lo, d_kall, d_Kg, m2,
                                                                                   nnodes, d_k, d_sumbg);
        PG_KERNEL_CHECK(ctx);
        std::vector<int> ones((size_t)G, 1);
        PG_TRY(h2d(d_restart, ones.data(), (size_t)G * 4));
        PG_TRY(h2d(d_state, hstate.data(), (size_t)G * sizeof(int2)));
        PG_TRY(h2d(d_beta, dzeros.data(), (size_t)G * 8));
        w.nnodes = nnodes;
        w.nblk = nblk;
        w.npb = npb;
        w.blk = d_blk;
        w.no = d_no;
        w.ng = d_ng;
        w.fb = d_fb;
        w.nb = d_nb;
        w.gid = d_gid;
        w.lay = lay;
        w.k = d_k;
        w.sumbg = d_sumbg;
        w.m2 = m2;
        w.stopmode = opts->stop;
        w.tol = tol;
        w.max_iter = max_iter;
        w.ngroups = G;
        w.state = d_state;
        w.restart = d_restart;
        w.iters = d_iters;
        w.beta = d_beta;
        w.lam = d_lam;
        w.vn = d_vn;
        w.vres = d_vres;
        w.rho = d_rho;

        // pass state per group: 0 first pass, 1 shifted pass, 2 finished
        std::vector<int> pass((size_t)G, 0), list;
        std::vector<double> lam_total((size_t)G, 0.0), hbeta((size_t)G, 0.0);
        mod_start<<<(unsigned)nblk, TPB, 0, st>>>(w, 0);
        PG_KERNEL_CHECK(ctx);
        const size_t lds = gather ? 0 : pgdev::sp_lds(lay.cap);
        const auto iter_fn = gather ? (lay.val ? mod_iter<true, true> : mod_iter<false, true>)
                                    : (lay.val ? mod_iter<true, false> : mod_iter<false, false>);
        if (!gather)
            PG_HIP(ctx, hipFuncSetAttribute((const void *)iter_fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        int it = 0, running = G;
        std::vector<double> hlam((size_t)G);
        while (running > 0) {
            for (int q = 0; q < BATCH; q++) iter_fn<<<(unsigned)nblk, TPB, lds, st>>>(w, it + q);
            it += BATCH;
            PG_KERNEL_CHECK(ctx);
            PG_HIP(ctx, hipMemcpyAsync(hstate.data(), d_state, (size_t)G * sizeof(int2), hipMemcpyDeviceToHost, st));
            PG_HIP(ctx, hipStreamSynchronize(st));
            list.clear();
            for (int g = 0; g < G; g++)
                if (pass[g] < 2 && hstate[g].x) list.push_back(g);
            if (list.empty()) continue;
            const int m = (int)list.size();
            PG_TRY(h2d(d_list, list.data(), (size_t)m * 4));
            mod_lambda<<<(unsigned)m, TPB, 0, st>>>(w, d_list);
            PG_KERNEL_CHECK(ctx);
            PG_HIP(ctx, hipMemcpyAsync(hlam.data(), d_lam, (size_t)G * 8, hipMemcpyDeviceToHost, st));
            PG_HIP(ctx, hipStreamSynchronize(st));
            std::vector<int> restart;
            for (int g : list) {
                const double lam = hlam[g];
                if (pass[g] == 0) {
                    lam_total[g] = lam;
                    // shift rule: groups above 25000 nodes use lambda < -0.01
                    // (modularity_GPU.cu:369), smaller ones lambda < 0
                    // (Modularity_CPU.cpp:183)
                    const bool shift = ng[g] > 25000 ? (lam < -0.01) : (lam < 0.0);
                    if (shift) {
                        pass[g] = 1;
                        restart.push_back(g);
                        continue;
                    }
                } else {
                    lam_total[g] += lam;
                }
                pass[g] = 2;
                running--;
            }
            if (!restart.empty()) {
                // second pass on B + beta I, beta = -lambda, from the start vector
                // no iteration ran since hstate was read: it is the device state
                std::vector<int> rflag((size_t)G, 0);
                for (int g : restart) {
                    hbeta[g] = -lam_total[g];
                    hstate[g] = make_int2(0, it);
                    rflag[g] = 1;
                }
                PG_TRY(h2d(d_restart, rflag.data(), (size_t)G * 4));
                mod_start<<<(unsigned)nblk, TPB, 0, st>>>(w, it);
                PG_KERNEL_CHECK(ctx);
                PG_TRY(h2d(d_beta, hbeta.data(), (size_t)G * 8));
                PG_TRY(h2d(d_state, hstate.data(), (size_t)G * sizeof(int2)));
                PG_HIP(ctx, hipStreamSynchronize(st));
            }
        }
        std::vector<double> hv((size_t)nnodes);
        PG_HIP(ctx, hipMemcpyAsync(hv.data(), d_vres, (size_t)nnodes * 8, hipMemcpyDeviceToHost, st));
        PG_HIP(ctx, hipStreamSynchronize(st));
        if (trace) {
            std::vector<int> hits((size_t)G);
            PG_HIP(ctx, hipMemcpy(hits.data(), d_iters, (size_t)G * 4, hipMemcpyDeviceToHost));
            int mx = 0, big = 0;
            for (int g = 0; g < G; g++) {
                mx = std::max(mx, hits[g]);
                big = std::max(big, ng[g]);
            }
            const double secs = std::chrono::duration<double>(std::chrono::steady_clock::now() - wave_t0).count();
            std::fprintf(stderr, "pg_modularity wave %d: rounds %d..%d, %d nodes (largest group %d), "
                         "%d launched iterations, max %d in one pass, %.3f s\n",
                         nwave, lo, hi - 1, nnodes, big, it, mx, secs);
        }
        nwave++;

        // bookkeeping in round order
        for (int g = 0; g < G; g++) {
            const int round = lo + g;
            if (ng[g] == 0) continue;
            nrounds++;
            const double lam = lam_total[g];
            const double *gv = hv.data() + no[g];
            if (round == 0) {
                if (lambda0) *lambda0 = lam;
                if (eig0) {
                    std::vector<double> e0((size_t)n, 0.0);
                    for (int a = 0; a < ng[g]; a++) e0[gid[no[g] + a]] = gv[a];
                    if (pg_is_device_ptr(eig0)) PG_HIP(ctx, hipMemcpy(eig0, e0.data(), (size_t)n * 8, hipMemcpyHostToDevice));
                    else std::memcpy(eig0, e0.data(), (size_t)n * 8);
                }
            }
            long long sp = 0, sn = 0;
            for (int a = 0; a < ng[g]; a++) {
                sp += gv[a] > 0;
                sn += gv[a] <= 0;
            }
            const bool split = lam > 0.01 && sp > 1 && sn > 1;  // LAMBDA, MIN_GROUP
            if (split) {
                for (int a = 0; a < ng[g]; a++)
                    res[gid[no[g] + a]] = maxr + 1 + (gv[a] * ((double)(sp - sn) + 0.5) <= 0);
                maxr += 2;
            } else {
                adj[round] = index++;
            }
        }
        lo = hi;
    }
    std::vector<int> lab((size_t)n);
    for (int i = 0; i < n; i++) lab[i] = adj[res[i]];
    if (pg_is_device_ptr(labels)) PG_HIP(ctx, hipMemcpy(labels, lab.data(), (size_t)n * 4, hipMemcpyHostToDevice));
    else std::memcpy(labels, lab.data(), (size_t)n * 4);
    if (q) {
        // W modularity_GPU.cu:500-509 with the same k and m convention
        int maxl = 0;
        for (int i = 0; i < n; i++) maxl = std::max(maxl, lab[i]);
        std::vector<double> kc((size_t)maxl + 2, 0.0), inside((size_t)n);
        double in = 0.0;
        if (n > 0) {
            PG_HIP(ctx, hipMemcpyAsync(d_res, lab.data(), (size_t)n * 4, hipMemcpyHostToDevice, st));
            mod_inside<<<(unsigned)pg_cdiv(n, 4), 256, 0, st>>>(drow, dcol, kmode == PG_MOD_BINARY_K ? nullptr : dval,
                                                                d_res, n, d_in);
            PG_KERNEL_CHECK(ctx);
            PG_HIP(ctx, hipMemcpyAsync(inside.data(), d_in, (size_t)n * 8, hipMemcpyDeviceToHost, st));
            PG_HIP(ctx, hipStreamSynchronize(st));
        }
        for (int i = 0; i < n; i++) {
            kc[lab[i]] += k[i];
            in += inside[i];
        }
        double s2 = 0.0;
        for (double x : kc) s2 += x * x;
        *q = m2 > 0.0 ? (in - s2 / m2) / m2 : 0.0;
    }
    if (rounds) *rounds = nrounds;
    return PG_OK;
}
