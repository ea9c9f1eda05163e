// efficiency.hip -- binary nodal efficiency and characteristic path length
// from all-pairs hop counts (U/BFS_MulCPU/BFS_MulCPU/APSP_BFS.cpp:100-192),
// MI355X (gfx950).
//
// The reference fills a dense n x n float hop matrix with one queue BFS per
// source and then walks it.  Here the hop counts never exist as a matrix:
//
//  * Bit-parallel BFS.  A batch of S sources (S a multiple of 4096) gives every
//    vertex S/64 visited words, one bit per source.  Level d -> d+1 is one
//    pull launch: one wave per (vertex w, 64-word chunk), lane k owns word k of
//    the chunk and ORs word k of every neighbour's visited set (512 contiguous
//    bytes per neighbour per wave), stopping as soon as the bits w still lacks
//    are all found.  New bits are the sources at distance exactly d+1.  A
//    source that reached no vertex at one level is finished: w no longer looks
//    for it (else every level would scan every row for the sources of other
//    components).
//  * Bit-sliced levels.  Bit b of the level at which (w, s) is reached is
//    OR-ed into plane b, so a batch keeps ceil(log2(depth+1)) planes of S/8
//    bytes per vertex instead of a byte or a float per pair.  Planes are
//    allocated as the depth grows.
//  * Ordered sums.  One lane per source adds 1.0f / d(s, j) in FP32 over j =
//    0..n-1 in order -- the reference's precision and order, so e_s is
//    bit-identical -- while other waves of its work-group rebuild the distances
//    from the planes, and others add (double)(1.0f / d) for j > s into the
//    source's FP64 share of the Lp sum.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "pg_flag.hpp"
#include "pg_internal.hpp"

namespace {

typedef unsigned long long u64;

constexpr int MAXPLANES = 31;  // levels < 2^31
constexpr int LEVEL_GROUP = 4;  // level launches per host progress check

struct Planes {
    u64 *p[MAXPLANES];
};

// visited words of a batch: vis[v * W + k]; sources base + 64k + b
__global__ void eff_init(int n, int W, int base, int nsrc, u64 *__restrict__ vis, u64 *__restrict__ found)
{
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < W) found[t] = 0ull;
    if (t >= (long long)n * W) return;
    const int v = (int)(t / W), k = (int)(t % W);
    const int lo = 64 * k;
    u64 x;
    if (lo >= nsrc) x = ~0ull;                // every bit an absent source
    else if (nsrc - lo >= 64) x = 0ull;
    else x = ~0ull << (nsrc - lo);
    const int own = v - base;
    if (own >= 0 && own < nsrc && (own >> 6) == k) x |= 1ull << (own & 63);
    vis[t] = x;
}

__global__ void eff_zero(long long count, u64 *__restrict__ p)
{
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < count) p[t] = 0ull;
}

// The sources that found a vertex at this level, collected by words; the load
// keeps most waves' atomics away once a word is full.
__device__ __forceinline__ void mark_found(u64 *f, u64 nb)
{
    if (nb & ~__hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) atomicOr(f, nb);
}

// Level d -> d+1, d >= 1.  found holds three levels' source words: level d's
// (written by the launch before), level d + 1's (cleared there, collected
// here), and level d + 2's, cleared here.  chg[d & 1][v][c]: the words of chunk c
// in which v got new bits at level d + 1; a neighbour matters only if it
// changed in a word that w still looks for, since w took everything older at
// the level before (a far source keeps a bit open in almost every row for
// many levels, and each of those levels read 512 bytes of every neighbour).
// n = 25,218, 6.4 M entries, depth 10: 8.5 ms over the levels (22.6 ms), of
// which levels 1 and 2, which read nearly every neighbour, take 2.85 ms each.
// prog[d] is raised when a wave found new bits; a launch whose previous level
// found none returns at once (the BFS has ended).  Atomics on a line go one
// after the other, about 10 ns each, and up to 12,288 vertices the found words
// are few lines: there the waves of a work-group with the same chunk mark once
// (a ring of 1,000: 9.2 us a level, 24.6 with an atomic per wave and word).
__global__ __launch_bounds__(256) void eff_level(const int *__restrict__ row, const int *__restrict__ col, int n,
                                                 int W, int d, const u64 *__restrict__ visA,
                                                 u64 *__restrict__ visB, Planes planes, int nplanes,
                                                 u64 *__restrict__ found, u64 *__restrict__ chg,
                                                 unsigned *__restrict__ prog)
{
    if (prog[d - 1] == 0u) return;
    const int lane = threadIdx.x & 63;
    const int chunks = W >> 6;
    const int wv = threadIdx.x >> 6;
    const long long wid = (long long)blockIdx.x * 4 + wv;
    if (wid < chunks) found[((d + 1) % 3) * W + wid * 64 + lane] = 0ull;
    const bool live = wid < (long long)n * chunks;
    if (!live && chunks >= 4) return;
    const int w = __builtin_amdgcn_readfirstlane(live ? (int)(wid / chunks) : 0);
    const int c = __builtin_amdgcn_readfirstlane((int)(wid % chunks));
    const int k = (c << 6) + lane;
    const u64 vis = live ? visA[(size_t)w * W + k] : ~0ull;
    const u64 need = ~vis & found[((d - 1) % 3) * W + k];
    const u64 words = __ballot(need != 0);  // words of the chunk w still looks for
    const u64 *cin = chg + (size_t)((d - 1) & 1) * n * chunks + c;
    u64 acc = 0;
    if (words) {
        const int a = row[w], b = row[w + 1];
        bool done = false;
        for (int base = a; base < b && !done; base += 64) {
            int v = 0;
            u64 m = 0;
            if (base + lane < b) {
                v = col[base + lane];
                m = cin[(size_t)v * chunks] & words;
            }
            u64 any = __ballot(m != 0);
            while (any && !done) {
                u64 x = 0;
#pragma unroll
                for (int q = 0; q < 8; q++) {
                    if (any == 0) break;
                    const int vv = __builtin_amdgcn_readlane(v, (int)__builtin_ctzll(any));
                    any &= any - 1;
                    if (need) x |= visA[(size_t)vv * W + k];
                }
                acc |= x;
                done = __all((acc & need) == need);
            }
        }
    }
    u64 nb = acc & need;
    if (live) visB[(size_t)w * W + k] = vis | nb;
    if (nb) {
        const unsigned lv = (unsigned)d + 1u;
        for (int b = 0; b < nplanes; b++)
            if ((lv >> b) & 1u) planes.p[b][(size_t)w * W + k] |= nb;
    }
    u64 fresh = __ballot(nb != 0);
    if (live && lane == 0) chg[(size_t)(d & 1) * n * chunks + (size_t)w * chunks + c] = fresh;
    if (chunks < 4) {
        // the waves with the same chunk mark as one
        __shared__ u64 sf[4][64];
        sf[wv][lane] = nb;
        __syncthreads();
        if (wv >= chunks) return;
        for (int q = wv + chunks; q < 4; q += chunks) nb |= sf[q][lane];
        fresh = __ballot(nb != 0);
    }
    if (nb) mark_found(&found[(d % 3) * W + k], nb);
    if (lane == 0 && fresh) pgdev::raise(&prog[d]);
}

// Level 0 -> 1 from the column indices alone: the sources at distance 1 from
// w are its neighbours inside the batch.  One wave per (w, 64-word chunk); the
// chunk's 4096 sources are a contiguous column range of w's sorted row, found
// from a sampled ballot and read 64 entries at a time, each such neighbour
// setting its bit in the LDS word of the lane owning it -- no neighbour
// visited words are read.
__global__ __launch_bounds__(256) void eff_level0(const int *__restrict__ row, const int *__restrict__ col, int n,
                                                  int W, int base, const u64 *__restrict__ visA,
                                                  u64 *__restrict__ visB, Planes planes,
                                                  u64 *__restrict__ found, u64 *__restrict__ chg,
                                                 unsigned *__restrict__ prog)
{
    __shared__ u64 sbits[4][64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int chunks = W >> 6;
    const long long wid = (long long)blockIdx.x * 4 + wv;
    if (wid < chunks) found[W + wid * 64 + lane] = 0ull;
    if (wid >= (long long)n * chunks) return;
    const int w = __builtin_amdgcn_readfirstlane((int)(wid / chunks));
    const int c = __builtin_amdgcn_readfirstlane((int)(wid % chunks));
    const int k = (c << 6) + lane;
    const long long v0 = (long long)base + 4096ll * c, v1 = v0 + 4096;
    const int a = row[w], b = row[w + 1], dw = b - a;
    // a start at or before the first column >= v0: 64 evenly spaced samples
    // and a ballot (the loop below filters v >= v0 itself)
    int start = b;
    if (dw > 0) {
        const int ps = a + (int)(((long long)lane * dw) >> 6);  // < b
        const unsigned long long m = __ballot(col[ps] >= v0);
        const int f = m ? __builtin_ctzll(m) : 64;
        start = f == 0 ? a : a + (int)(((long long)(f - 1) * dw) >> 6);
    }
    // the chunk's neighbours, 64 at a time, each OR-ed into the LDS word of
    // the lane owning it
    sbits[wv][lane] = 0ull;
    __threadfence_block();
    for (int e0 = start; e0 < b; e0 += 64) {
        const int e = e0 + lane;
        const long long v = e < b ? (long long)col[e] : v1;
        if (v >= v0 && v < v1) {
            const int rel = (int)(v - v0);
            atomicOr(&sbits[wv][rel >> 6], 1ull << (rel & 63));
        }
        if (__ballot(e < b && v >= v1)) break;  // columns ascend: the chunk is done
    }
    __threadfence_block();
    const u64 acc = atomicOr(&sbits[wv][lane], 0ull);
    const u64 vis = visA[(size_t)w * W + k];
    const u64 nb = acc & ~vis;
    visB[(size_t)w * W + k] = vis | nb;
    if (nb) {
        planes.p[0][(size_t)w * W + k] |= nb;
        mark_found(&found[k], nb);
    }
    const u64 fresh = __ballot(nb != 0);
    if (lane == 0) {
        chg[(size_t)w * chunks + c] = fresh;
        if (fresh) pgdev::raise(&prog[0]);
    }
}

// Work-group k sums 64 sources (word k of the batch).  The FP32 sum of a source
// is a chain of n dependent adds, so one wave does nothing else: it adds
// values that SUM_PROD waves put into LDS 64 vertices at a time (lane = vertex,
// the source's bit of each plane -> level -> 1 / level from a table; rows of a
// tile padded to 68 floats, so that lane = source then reads four in one
// conflict-free access), and two waves take the FP64 shares of alternate
// tiles.  Two sets of tiles, one barrier per round of 64 SUM_PROD vertices.
// n = 25,218, four planes: 0.84 ms (4.4 ms with one wave per 64 sources that
// did all of it).
constexpr int SUM_PROD = 4, SUM_TPB = 64 * (3 + SUM_PROD), SUM_LD = 68;
constexpr size_t SUM_LDS = (size_t)2 * SUM_PROD * 64 * SUM_LD * 4 + 256 * 4;
template <int NP>
__global__ __launch_bounds__(SUM_TPB) void eff_sum(int n, int W, int base, int nsrc, Planes planes,
                                                   float *__restrict__ eff, double *__restrict__ lpp,
                                                   int *__restrict__ flags)
{
    extern __shared__ __align__(16) float sm[];
    __shared__ double dpart[64];
    __shared__ int rpart[64];
    float *rtab = sm + 2 * SUM_PROD * 64 * SUM_LD;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int k = blockIdx.x;
    const int s = base + 64 * k + lane;
    constexpr bool TAB = NP <= 8;
    if (TAB && threadIdx.x < (1 << (TAB ? NP : 0))) rtab[threadIdx.x] = threadIdx.x ? 1.0f / (float)(int)threadIdx.x : 0.0f;
    const int rounds = (n + 64 * SUM_PROD - 1) / (64 * SUM_PROD);
    const int p = wv - 3;  // producer
    u64 w[NP];
    auto fetch = [&](int r) {
        const int j = (r * SUM_PROD + p) * 64 + lane;
#pragma unroll
        for (int b = 0; b < NP; b++) w[b] = j < n ? planes.p[b][(size_t)j * W + k] : 0ull;
    };
    if (p >= 0) fetch(0);
    float acc = 0.0f;
    double dacc = 0.0;
    int reached = 0;
    __syncthreads();
    for (int r = 0; r <= rounds; r++) {
        if (p >= 0) {
            if (r < rounds) {
                float *t = sm + ((r & 1) * SUM_PROD + p) * 64 * SUM_LD + lane;
                uint32_t lo[NP], hi[NP];
#pragma unroll
                for (int b = 0; b < NP; b++) {
                    lo[b] = (uint32_t)w[b];
                    hi[b] = (uint32_t)(w[b] >> 32);
                }
                if (r + 1 < rounds) fetch(r + 1);
#pragma unroll 8
                for (int q = 0; q < 32; q++) {
                    int l0 = 0, l1 = 0;
#pragma unroll
                    for (int b = 0; b < NP; b++) {
                        l0 |= (int)((lo[b] >> q) & 1u) << b;
                        l1 |= (int)((hi[b] >> q) & 1u) << b;
                    }
                    if (TAB) {
                        t[q * SUM_LD] = rtab[l0];
                        t[(q + 32) * SUM_LD] = rtab[l1];
                    } else {
                        t[q * SUM_LD] = l0 ? 1.0f / (float)l0 : 0.0f;
                        t[(q + 32) * SUM_LD] = l1 ? 1.0f / (float)l1 : 0.0f;
                    }
                }
            }
        } else if (r > 0) {
            const float *t0 = sm + ((r - 1) & 1) * SUM_PROD * 64 * SUM_LD + lane * SUM_LD;
            if (wv == 0) {
                for (int q = 0; q < SUM_PROD; q++) {
                    const float4 *t = (const float4 *)(t0 + q * 64 * SUM_LD);
#pragma unroll
                    for (int j = 0; j < 16; j++) {
                        const float4 v = t[j];
                        acc += v.x;
                        acc += v.y;
                        acc += v.z;
                        acc += v.w;
                    }
                }
            } else {
                for (int q = wv - 1; q < SUM_PROD; q += 2) {
                    const float4 *t = (const float4 *)(t0 + q * 64 * SUM_LD);
                    const int j0 = ((r - 1) * SUM_PROD + q) * 64 - s;  // j > s: j - s > 0
#pragma unroll 4
                    for (int j = 0; j < 16; j++) {
                        const float4 v = t[j];
                        reached += (v.x != 0.0f) + (v.y != 0.0f) + (v.z != 0.0f) + (v.w != 0.0f);
                        dacc += j0 + 4 * j > 0 ? (double)v.x : 0.0;
                        dacc += j0 + 4 * j + 1 > 0 ? (double)v.y : 0.0;
                        dacc += j0 + 4 * j + 2 > 0 ? (double)v.z : 0.0;
                        dacc += j0 + 4 * j + 3 > 0 ? (double)v.w : 0.0;
                    }
                }
            }
        }
        __syncthreads();
    }
    if (wv == 2) {
        dpart[lane] = dacc;
        rpart[lane] = reached;
    }
    __syncthreads();
    if (64 * k + lane >= nsrc) return;
    if (wv == 0) {
        const float e = acc / (float)(n - 1);
        eff[s] = e;
        if (e == 0.0f) atomicAdd(&flags[0], 1);
    } else if (wv == 1) {
        lpp[s] = dacc + dpart[lane];
        if (reached + rpart[lane] < n - 1) atomicOr(&flags[1], 1);
    }
}

template <int NP>
hipError_t launch_sum(hipStream_t st, int n, int W, int base, int nsrc, const Planes &pl, float *eff, double *lpp,
                      int *flags)
{
    const hipError_t e = hipFuncSetAttribute((const void *)eff_sum<NP>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                             (int)SUM_LDS);
    if (e != hipSuccess) return e;
    eff_sum<NP><<<(unsigned)((nsrc + 63) / 64), SUM_TPB, SUM_LDS, st>>>(n, W, base, nsrc, pl, eff, lpp, flags);
    return hipGetLastError();
}

typedef hipError_t (*SumFn)(hipStream_t, int, int, int, int, const Planes &, float *, double *, int *);

SumFn sum_fn(int np)
{
    static const SumFn t[MAXPLANES + 1] = {
        launch_sum<1>,  launch_sum<1>,  launch_sum<2>,  launch_sum<3>,  launch_sum<4>,  launch_sum<5>,
        launch_sum<6>,  launch_sum<7>,  launch_sum<8>,  launch_sum<9>,  launch_sum<10>, launch_sum<11>,
        launch_sum<12>, launch_sum<13>, launch_sum<14>, launch_sum<15>, launch_sum<16>, launch_sum<17>,
        launch_sum<18>, launch_sum<19>, launch_sum<20>, launch_sum<21>, launch_sum<22>, launch_sum<23>,
        launch_sum<24>, launch_sum<25>, launch_sum<26>, launch_sum<27>, launch_sum<28>, launch_sum<29>,
        launch_sum<30>, launch_sum<31>};
    return t[np];
}

int bit_width(unsigned x)
{
    int b = 0;
    while (x) {
        b++;
        x >>= 1;
    }
    return b;
}

// Sources per batch: all of them when the visited words and four planes fit
// in the budget, else the largest multiple of 4096 that does.
int batch_sources(int n, size_t budget)
{
    const long long all = pg_cdiv(n, 4096) * 4096;
    const double per_source = (double)n / 8.0 * 6.0;
    long long fit = (long long)((double)budget / per_source) / 4096 * 4096;
    fit = std::max<long long>(fit, 4096);
    return (int)std::min(all, fit);
}

}  // namespace

extern "C" pg_status pg_bfs_efficiency(pg_ctx *ctx, const int32_t *row, const int32_t *col, int32_t n,
                                       int64_t nnz, float *eff, double *lp, int32_t *isolated,
                                       int32_t *unconnected)
{
    if (!ctx) return PG_EINVAL;
    PG_HIP(ctx, hipSetDevice(ctx->device));
    PG_TRY(pg_check_csr_args(ctx, row, col, n, nnz));
    if (n < 1) return pg_fail(ctx, PG_EINVAL, "n must be >= 1");
    const int *drow, *dcol;
    PG_TRY(pg_in(ctx, row, (size_t)n + 1, "in.row", &drow));
    PG_TRY(pg_in(ctx, col, (size_t)nnz, "in.col", &dcol));
    hipStream_t st = ctx->stream;

    const char *env = std::getenv("PAGANI_EFF_BATCH");
    int S = batch_sources(n, (size_t)4 << 30);
    if (env && std::atoi(env) > 0) S = (int)std::min<long long>(pg_cdiv(std::atoi(env), 4096) * 4096, S);
    const int W = S / 64;
    const size_t words = (size_t)n * W;
    u64 *va, *vb, *found, *chg;
    unsigned *prog;
    float *deff;
    double *lpp;
    int *flags;
    PG_TRY(pg_bufT(ctx, "eff.visA", words, &va));
    PG_TRY(pg_bufT(ctx, "eff.visB", words, &vb));
    PG_TRY(pg_bufT(ctx, "eff.found", (size_t)3 * W, &found));
    PG_TRY(pg_bufT(ctx, "eff.chg", (size_t)2 * n * (W / 64), &chg));
    PG_TRY(pg_bufT(ctx, "eff.prog", (size_t)n + LEVEL_GROUP + 2, &prog));
    PG_TRY(pg_bufT(ctx, "eff.lpp", (size_t)n, &lpp));
    PG_TRY(pg_bufT(ctx, "eff.flags", 2, &flags));
    PG_TRY(pg_out(ctx, eff, (size_t)n, "out.eff", &deff));
    if (!deff) PG_TRY(pg_bufT(ctx, "eff.scratch", (size_t)n, &deff));
    PG_HIP(ctx, hipMemsetAsync(flags, 0, 8, st));
    PG_TRY(pg_validate_csr(ctx, drow, dcol, n, nnz, true));

    Planes pl = {};
    int nplanes = 0;
    auto grow = [&](int want) -> pg_status {
        for (; nplanes < want; nplanes++) {
            char name[32];
            std::snprintf(name, sizeof name, "eff.plane%d", nplanes);
            PG_TRY(pg_bufT(ctx, name, words, &pl.p[nplanes]));
            eff_zero<<<(unsigned)pg_cdiv((long long)words, 256), 256, 0, st>>>((long long)words, pl.p[nplanes]);
        }
        return PG_OK;
    };

    for (int base = 0; base < n; base += S) {
        const int nsrc = std::min(S, n - base);
        for (int b = 0; b < nplanes; b++)
            eff_zero<<<(unsigned)pg_cdiv((long long)words, 256), 256, 0, st>>>((long long)words, pl.p[b]);
        PG_HIP(ctx, hipMemsetAsync(prog, 0, ((size_t)n + LEVEL_GROUP + 2) * 4, st));
        eff_init<<<(unsigned)pg_cdiv((long long)words, 256), 256, 0, st>>>(n, W, base, nsrc, va, found);
        PG_KERNEL_CHECK(ctx);
        const unsigned blocks = (unsigned)pg_cdiv((long long)n * (W / 64), 4);
        int depth = -1;
        for (int d = 0; depth < 0; d += LEVEL_GROUP) {
            if (d > n) return pg_fail(ctx, PG_EDEVICE, "BFS did not converge");
            const int top = std::min(d + LEVEL_GROUP, n + 1);  // levels reachable by this group
            if (bit_width((unsigned)top) > MAXPLANES) return pg_fail(ctx, PG_ENOTSUP, "graph too deep");
            PG_TRY(grow(bit_width((unsigned)top)));
            for (int q = 0; q < LEVEL_GROUP; q++) {
                if (d + q == 0)
                    eff_level0<<<blocks, 256, 0, st>>>(drow, dcol, n, W, base, va, vb, pl, found, chg, prog);
                else
                    eff_level<<<blocks, 256, 0, st>>>(drow, dcol, n, W, d + q, va, vb, pl, nplanes, found, chg, prog);
                std::swap(va, vb);
            }
            PG_KERNEL_CHECK(ctx);
            unsigned h[LEVEL_GROUP];
            PG_HIP(ctx, hipMemcpyAsync(h, prog + d, sizeof h, hipMemcpyDeviceToHost, st));
            PG_HIP(ctx, hipStreamSynchronize(st));
            for (int q = 0; q < LEVEL_GROUP && depth < 0; q++)
                if (h[q] == 0) depth = d + q;  // deepest level present
        }
        const int np = std::max(1, bit_width((unsigned)depth));
        PG_HIP(ctx, sum_fn(np)(st, n, W, base, nsrc, pl, deff, lpp, flags));
    }
    PG_TRY(pg_out_finish(ctx, eff, deff, (size_t)n));
    std::vector<double> h((size_t)n);
    int hf[2] = {0, 0};
    PG_HIP(ctx, hipMemcpyAsync(h.data(), lpp, (size_t)n * 8, hipMemcpyDeviceToHost, st));
    PG_HIP(ctx, hipMemcpyAsync(hf, flags, 8, hipMemcpyDeviceToHost, st));
    PG_HIP(ctx, hipStreamSynchronize(st));
    if (lp) {
        double x = 0.0;
        for (int s = 0; s < n; s++) x += h[(size_t)s];
        x /= (double)n;
        x /= (double)(n - 1);
        *lp = 1 / x / 2;
    }
    if (isolated) *isolated = hf[0];
    if (unconnected) *unconnected = hf[1];
    return PG_OK;
}

namespace {
// bad = 1 unless row is non-decreasing from row[0] = 0 to row[n] = nnz and
// every col is in [0, n); sorted: also strictly ascending columns inside each
// row.  One wave per row; a row whose bounds fall outside [0, nnz] is flagged
// before any of its columns is read, so the check itself stays in bounds.
// col == nullptr checks the row offsets only.
__global__ __launch_bounds__(256) void csr_validate(const int *__restrict__ row, const int *__restrict__ col, int n,
                                                    long long nnz, int sorted, int *__restrict__ bad)
{
    const long long w = ((long long)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int lane = threadIdx.x & 63;
    bool ok = true;
    if (w < n) {
        const long long a = row[w], b = row[w + 1];
        ok = a >= 0 && a <= b && b <= nnz;
        if (ok && col) {
            // four loads in flight; a column's left neighbour comes from the
            // lane before, the batch before, or nowhere at the row's start
            int prev = -1;  // last column of the batch before
            for (long long e0 = a; e0 < b; e0 += 256) {
                int c[4];
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const long long e = e0 + 64 * u + lane;
                    c[u] = e < b ? col[e] : INT_MAX;
                }
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const bool in = e0 + 64 * u + lane < b;
                    int left = __shfl_up(c[u], 1);
                    if (lane == 0) left = prev;
                    ok = ok && (!in || (c[u] >= 0 && c[u] < n && !(sorted && left >= c[u])));
                    prev = __shfl(c[u], 63);
                }
            }
        }
    }
    if (w == 0 && lane == 0) ok = ok && row[0] == 0 && (long long)row[n] == nnz;
    if (!ok) *(volatile int *)bad = 1;
}
}  // namespace

void pg_validate_launch(pg_ctx *ctx, const int32_t *drow, const int32_t *dcol, int32_t n, int64_t nnz, bool sorted,
                        int *bad)
{
    const long long waves = std::max<long long>(n, 1);
    csr_validate<<<(unsigned)pg_cdiv(waves, 4), 256, 0, ctx->stream>>>(drow, dcol, n, nnz, sorted ? 1 : 0, bad);
}

pg_status pg_malformed(pg_ctx *ctx, bool sorted)
{
    return pg_fail(ctx, PG_EFORMAT, "malformed CSR (row not 0..nnz non-decreasing, col out of range%s)",
                   sorted ? " or columns not ascending in a row" : "");
}

pg_status pg_validate_csr(pg_ctx *ctx, const int32_t *drow, const int32_t *dcol, int32_t n, int64_t nnz,
                          bool sorted)
{
    // the flag is the context's pinned word: no clearing launch, no copy
    volatile int *bad = &pg_check(ctx)->bad;
    *bad = 0;
    pg_validate_launch(ctx, drow, dcol, n, nnz, sorted, (int *)bad);
    PG_KERNEL_CHECK(ctx);
    PG_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return *bad ? pg_malformed(ctx, sorted) : PG_OK;
}
