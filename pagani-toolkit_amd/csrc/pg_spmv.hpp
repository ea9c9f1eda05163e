// pg_spmv.hpp -- sparse matrix times FP64 vector for the power iterations
// (modularity, eigenvector centrality), MI355X (gfx950).
//
// An FP64 gather straight from L2 costs the texture addresser one line per
// lane (64 clocks per 64 entries), so the vector is staged in LDS, SP_SEG
// entries (128 KB of the CU's 160 KB) at a time, and gathered there.  Rows are
// split by segment into parts, a part's entries stored as 16-bit
// segment-relative columns (and FP32 weights) in groups of four, its last
// group filled with the index of a zero LDS slot (weight 0): one 8-byte load
// (and one of 16) brings a lane four entries, aligned and without bounds.  16
// lanes take a part, so a work-group of 1,024 threads works on 64 rows at once
// and a row of up to 256 entries has all its loads in flight.  Row i's parts
// start at group ceil(row[i] / 4) + i * nseg and follow each other: the
// fillers always fit before row i + 1's, so the layout needs no scan.
//
// Staging costs a work-group the whole vector, however few entries its rows
// have, and the layout a part per row and segment.  A sparse network (sp_gathers)
// keeps its entries in row order with 32-bit columns and gathers the vector
// from L2: memory in the entries and rows only, at any length of the vector.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>

namespace pgdev {

constexpr int SP_TPB = 1024;     // threads per work-group: 64 rows of 16 lanes
constexpr int SP_SEG = 16384;    // vector entries per LDS segment
constexpr int SP_ROWS = 1024;    // most rows per work-group
constexpr int SP_LOADS = SP_SEG / (2 * SP_TPB);  // 16-byte staging loads per thread

typedef double sp_d2u __attribute__((ext_vector_type(2), aligned(8)));

struct SpLayout {
    uint16_t *idx;  // groups of 4
    int *gcol;      // the gathered form's columns: row i's from place row[i] on
    float *val;     // the same places (NULL: every weight is 1)
    int2 *part;     // [rows][nseg]: first group, groups; gathered: [rows]: first entry, entries
    uint16_t *perm; // [rows]: a work-group's row of each of its slots, longest rows first
    int nseg, cap;  // segments of a row's vector (0: gathered); its entries per segment (the zero slot's index)
};

inline int sp_nseg(long long n) { return (int)std::max<long long>(1, (n + SP_SEG - 1) / SP_SEG); }
inline int sp_cap(long long n) { return (int)std::max<long long>(1, std::min<long long>(n, SP_SEG)); }
// entries of idx / val for nnz entries of n rows
inline size_t sp_room(long long n, long long nnz, int nseg)
{
    return 4 * ((size_t)(nnz + 3) / 4 + (size_t)n * nseg + 1);
}
// dynamic LDS: the segment, the zero slot
inline size_t sp_lds(int cap) { return ((size_t)cap + 1) * sizeof(double); }

// Gathered form for nnz entries of n rows in `blocks` work-groups: fewer than
// 3,000 entries per work-group and segment.  Microseconds of a modularity
// iteration, staged / gathered (random networks, unweighted or weighted), at
// this many of them: n = 2,000 7.9 / 6.8 at 320, 15.5 / 16.1 at 3,000 (two
// passes); 16,000 18.2 / 16.6 at 1,260, 9.4 / 9.3 at 3,150, 18.9 / 21.5 at
// 6,280; 58,000 28.7 / 12.2 at 1,130, 28.6 / 18.7 at 2,830, 57.6 / 58.9 at
// 5,660, 29.7 / 87.0 at 22,600; 200,000 176 / 32 at 1,200, 192 / 176 at 12,000;
// 1,000,000 2,800 / 81 at 165.  The staged form's group numbers are 32-bit: it is
// taken with nnz >= 3,000 n nseg / SP_ROWS at least, hence n * nseg + nnz / 4 <
// 0.6 nnz < 2^31.
constexpr long long SP_GATHER = 3000;
inline bool sp_gathers(long long n, long long nnz, long long blocks) { return nnz < SP_GATHER * blocks * sp_nseg(n); }

// Layout of rows a = 0 .. nrows - 1 by one wave each: row i = gid[a] (a itself
// when gid is NULL), its entries (i, j) with grp[j] == grp[i] (all when grp is
// NULL) at vector position loc[j] - base[grp[i] - grp0] (j itself).  Columns
// may come in any order: a pass per segment.  kin[a] (may be NULL): FP64 sum
// of the kept weights (their count with `count`).
static __global__ __launch_bounds__(256) void sp_build(const int *__restrict__ row, const int *__restrict__ col,
                                                const float *__restrict__ val, int nrows,
                                                const int *__restrict__ gid, const int *__restrict__ grp, int grp0,
                                                const int *__restrict__ base, const int *__restrict__ loc, SpLayout L,
                                                double *__restrict__ kin, int count)
{
    const int a = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (a >= nrows) return;
    const int i = gid ? gid[a] : a;
    const int r0 = row[i], r1 = row[i + 1];
    const int g = grp ? grp[i] : 0, b0 = grp ? base[g - grp0] : 0;
    int g0 = (int)(((long long)r0 + 3) / 4 + (long long)i * L.nseg);
    double k = 0.0;
    if (L.nseg == 0) {
        int have = 0;
        for (long long e0 = r0; e0 < r1; e0 += 64) {
            const long long e = e0 + lane;
            int p = -1;
            if (e < r1) {
                const int j = col[e];
                if (!grp || grp[j] == g) p = grp ? loc[j] - b0 : j;
            }
            const unsigned long long m = __ballot(p >= 0);
            if (p >= 0) {
                const int at = r0 + have + __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
                const float w = val ? val[e] : 1.0f;
                L.gcol[at] = p;
                if (L.val) L.val[at] = w;
                k += count ? 1.0 : (double)w;
            }
            have += __popcll(m);
        }
        if (lane == 0) L.part[a] = make_int2(r0, have);
    }
    for (int s = 0; s < L.nseg; s++) {
        int have = 0;
        for (long long e0 = r0; e0 < r1; e0 += 64) {
            const long long e = e0 + lane;
            int p = -1;
            if (e < r1) {
                const int j = col[e];
                if (!grp || grp[j] == g) p = (grp ? loc[j] - b0 : j) - s * SP_SEG;
            }
            const bool keep = p >= 0 && p < SP_SEG;
            const unsigned long long m = __ballot(keep);
            if (keep) {
                const int at = have + __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
                const float w = val ? val[e] : 1.0f;
                L.idx[4ll * g0 + at] = (uint16_t)p;
                if (L.val) L.val[4ll * g0 + at] = w;
                k += count ? 1.0 : (double)w;
            }
            have += __popcll(m);
        }
        const int ng = (have + 3) / 4;
        if (have + lane < 4 * ng) {
            L.idx[4ll * g0 + have + lane] = (uint16_t)L.cap;
            if (L.val) L.val[4ll * g0 + have + lane] = 0.0f;
        }
        if (lane == 0) L.part[(long long)a * L.nseg + s] = make_int2(g0, ng);
        g0 += ng;
    }
    if (kin) {
        for (int o = 32; o > 0; o >>= 1) k += __shfl_xor(k, o);
        if (lane == 0) kin[a] = k;
    }
}

// Row order of the work-groups: perm[a0 + rank] = row - a0 over the rows [a0, a0
// + nr) of one, by falling length (equal lengths in row order).  Four rows
// share a wave and wait for the longest of them; degrees of a thresholded
// network differ by ten times (weighted modularity of 14,011 nodes 43.7 ->
// 41.7 ms).  blk gives a0 and nr of work-group b.
template <class BlockRange>
__global__ __launch_bounds__(SP_TPB) void sp_order(const int *__restrict__ row, const int *__restrict__ gid,
                                                   BlockRange blk, uint16_t *__restrict__ perm)
{
    __shared__ int len[SP_ROWS];
    int a0, nr;
    blk(blockIdx.x, a0, nr);
    const int tid = threadIdx.x;
    if (tid < nr) {
        const int i = gid ? gid[a0 + tid] : a0 + tid;
        len[tid] = row[i + 1] - row[i];
    }
    __syncthreads();
    if (tid >= nr) return;
    const int mine = len[tid];
    int rank = 0;
    for (int q = 0; q < nr; q++) rank += len[q] > mine || (len[q] == mine && q < tid);
    perm[a0 + rank] = (uint16_t)tid;
}

// Sum over the caller's row of 16 lanes, in every lane (DPP rotations).
template <int N>
__device__ __forceinline__ double sp_ror(double x)
{
    const long long b = __double_as_longlong(x);
    const unsigned lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)b, 0x120 + N, 0xf, 0xf, true);
    const unsigned hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), 0x120 + N, 0xf, 0xf, true);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ double sp_sum16(double x)
{
    x += sp_ror<8>(x);
    x += sp_ror<4>(x);
    x += sp_ror<2>(x);
    x += sp_ror<1>(x);
    return x;
}

// NB groups of a part per lane (l = 0 .. 15), from group g on: 256 entries, 128
// where the weights' registers would spill.
template <bool W>
struct SpBatch {
    static constexpr int NB = W ? 2 : 4;
    uint2 c[NB];
    float4 w[NB];
    __device__ __forceinline__ void load(const SpLayout &L, int g, int end)
    {
        const uint2 *ix = (const uint2 *)L.idx;
        const float4 *wx = (const float4 *)L.val;
        const unsigned pad = (unsigned)L.cap * 0x10001u;
#pragma unroll
        for (int u = 0; u < NB; u++) {
            const bool in = g + 16 * u < end;
            c[u] = in ? ix[g + 16 * u] : make_uint2(pad, pad);
            if (W) w[u] = in ? wx[g + 16 * u] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
    }
    __device__ __forceinline__ double dot(const double *__restrict__ xs, double acc) const
    {
#pragma unroll
        for (int u = 0; u < NB; u++) {
            const double x0 = xs[c[u].x & 0xffffu], x1 = xs[c[u].x >> 16];
            const double x2 = xs[c[u].y & 0xffffu], x3 = xs[c[u].y >> 16];
            if (W) {
                acc = fma(x0, (double)w[u].x, acc);
                acc = fma(x1, (double)w[u].y, acc);
                acc = fma(x2, (double)w[u].z, acc);
                acc = fma(x3, (double)w[u].w, acc);
            } else {
                acc += (x0 + x1) + (x2 + x3);
            }
        }
        return acc;
    }
};

// Row sums of rows a0 .. a0 + nr - 1 (nr <= SP_ROWS) against x[0 .. len) into
// rowv[0 .. nr), behind a barrier; slot k is row a0 + perm[a0 + k].  A pass
// takes 64 slots, every other one in reverse, so that no wave has the longest
// rows of all passes.  xs: sp_lds(cap) of LDS; pt: SP_ROWS int2 of
// LDS.  Latency is what the loop hides: a segment's vector entries and part
// bounds are loaded into registers under the segment before it (the first
// under `between`, which the caller's own waits go into; it returns whether to
// go on, the same in every thread), and a part's entries under the part
// before it, a segment's first parts under the segment before and its own
// staging: their bounds are also loaded by the lanes that take them.
template <bool W, class F>
__device__ __forceinline__ bool sp_rows(const SpLayout &L, int a0, int nr, const double *__restrict__ x, int len,
                                        double *__restrict__ xs, int2 *__restrict__ pt, double *__restrict__ rowv,
                                        F &&between)
{
    const int tid = threadIdx.x, l = tid & 15, q = tid >> 4;
    const int2 *part = L.part + (long long)(a0 + (tid < nr ? (int)L.perm[a0 + tid] : 0)) * L.nseg;
    const int2 *first = L.part + (long long)(a0 + (q < nr ? (int)L.perm[a0 + q] : 0)) * L.nseg;
    sp_d2u v[SP_LOADS];
    int2 pn = make_int2(0, 0), pf = make_int2(0, 0);
    auto load = [&](int s) {
        const double *xb = x + (long long)s * SP_SEG;
        const int m = min(SP_SEG, len - s * SP_SEG);
#pragma unroll
        for (int u = 0; u < SP_LOADS; u++) {
            const int k = 2 * (tid + u * SP_TPB);
            v[u].x = 0.0;
            v[u].y = 0.0;
            if (k + 1 < m) v[u] = *(const sp_d2u *)(xb + k);
            else if (k < m) v[u].x = xb[k];
        }
        if (tid < nr) pn = part[s];
        if (q < nr) pf = first[s];
    };
    load(0);
    if (!between()) return false;
    SpBatch<W> b, c;
    int2 p = pf;
    b.load(L, p.x + l, p.x + p.y);
    for (int s = 0; s * SP_SEG < len; s++) {
        const int m = min(SP_SEG, len - s * SP_SEG);
        if (s > 0) __syncthreads();  // the previous segment's readers are done
#pragma unroll
        for (int u = 0; u < SP_LOADS; u++) {
            const int k = 2 * (tid + u * SP_TPB);
            if (k < m) xs[k] = v[u].x;
            if (k + 1 < m) xs[k + 1] = v[u].y;
        }
        if (tid == 0) xs[L.cap] = 0.0;
        if (tid < nr) pt[tid] = pn;
        __syncthreads();
        constexpr int Q = SP_TPB / 16;
        int r = q;  // this pass's slot, and the next's
        pf = make_int2(0, 0);
        if ((s + 1) * SP_SEG < len) load(s + 1);
        for (int k0 = 0; k0 < nr; k0 += Q) {
            const int rn = k0 + Q + ((k0 / Q) & 1 ? q : Q - 1 - q);
            const int end = p.x + p.y;
            double acc = 0.0;
            int g = p.x + l;
            constexpr int step = 16 * SpBatch<W>::NB;
            for (; g - l + step < end; g += step) {  // more of this part to come
                c.load(L, g + step, end);
                acc = b.dot(xs, acc);
                b = c;
            }
            if (k0 + Q < nr) p = rn < nr ? pt[rn] : make_int2(0, 0);
            else p = pf;
            c.load(L, p.x + l, p.x + p.y);
            acc = b.dot(xs, acc);
            b = c;
            acc = sp_sum16(acc);
            if (l == 0 && r < nr) rowv[r] = s > 0 ? rowv[r] + acc : acc;
            r = rn;
        }
    }
    __syncthreads();
    return true;
}

// Four entries of row part p (first entry, entries) per lane, from its entry k on.
template <bool W>
struct SpGather {
    int c[4];
    float w[4];
    __device__ __forceinline__ void load(const SpLayout &L, int2 p, int k)
    {
        const long long e = (long long)p.x + k;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const bool in = k + 16 * u < p.y;
            c[u] = in ? L.gcol[e + 16 * u] : -1;
            if (W) w[u] = in ? L.val[e + 16 * u] : 0.0f;
        }
    }
    __device__ __forceinline__ double dot(const double *__restrict__ x, double acc) const
    {
        double v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = c[u] >= 0 ? x[c[u]] : 0.0;
#pragma unroll
        for (int u = 0; u < 4; u++) acc = W ? fma(v[u], (double)w[u], acc) : acc + v[u];
        return acc;
    }
};

// sp_rows of the gathered form: x is read where it lies.  The entries of the
// next 64 slots are loaded under the look-ups of these.
template <bool W, class F>
__device__ __forceinline__ bool sp_rows_gather(const SpLayout &L, int a0, int nr, const double *__restrict__ x,
                                               int2 *__restrict__ pt, double *__restrict__ rowv, F &&between)
{
    const int tid = threadIdx.x, l = tid & 15, q = tid >> 4;
    int2 pn = make_int2(0, 0), p = make_int2(0, 0);
    if (tid < nr) pn = L.part[a0 + (int)L.perm[a0 + tid]];
    if (q < nr) p = L.part[a0 + (int)L.perm[a0 + q]];
    if (!between()) return false;
    SpGather<W> b, c;
    b.load(L, p, l);
    if (tid < nr) pt[tid] = pn;
    __syncthreads();
    constexpr int Q = SP_TPB / 16;
    int r = q;  // this pass's slot, and the next's
    for (int k0 = 0; k0 < nr; k0 += Q) {
        const int rn = k0 + Q + ((k0 / Q) & 1 ? q : Q - 1 - q);
        double acc = 0.0;
        for (int k = 64; k < p.y; k += 64) {  // more of this row to come
            c.load(L, p, k + l);
            acc = b.dot(x, acc);
            b = c;
        }
        p = rn < nr ? pt[rn] : make_int2(0, 0);
        c.load(L, p, l);
        acc = b.dot(x, acc);
        b = c;
        acc = sp_sum16(acc);
        if (l == 0 && r < nr) rowv[r] = acc;
        r = rn;
    }
    __syncthreads();
    return true;
}

// Either form.
template <bool W, bool GATHER, class F>
__device__ __forceinline__ bool sp_product(const SpLayout &L, int a0, int nr, const double *__restrict__ x, int len,
                                           double *__restrict__ xs, int2 *__restrict__ pt, double *__restrict__ rowv,
                                           F &&between)
{
    if constexpr (GATHER) return sp_rows_gather<W>(L, a0, nr, x, pt, rowv, between);
    else return sp_rows<W>(L, a0, nr, x, len, xs, pt, rowv, between);
}

// Q sums over the first nr threads of the work-group in a fixed order, written
// by thread k < Q to out[k]; red: SP_TPB / 64 * Q doubles.
template <int Q>
__device__ __forceinline__ void sp_block_sums(double (&v)[Q], int nr, double *__restrict__ red, double *__restrict__ out)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = (nr + 63) >> 6;
    if (w < nw) {
#pragma unroll
        for (int k = 0; k < Q; k++) {
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) v[k] += __shfl_xor(v[k], o);
            if (lane == 0) red[w * Q + k] = v[k];
        }
    }
    __syncthreads();
    if (threadIdx.x < Q) {
        double s = 0.0;
        for (int q = 0; q < nw; q++) s += red[q * Q + threadIdx.x];
        out[threadIdx.x] = s;
    }
}

// Sums of Q per-block partials part[f .. f + m)[Q], one wave per quantity, in
// a fixed order (every thread gets them); tot: Q doubles.
template <int Q>
__device__ __forceinline__ void sp_partials(const double *__restrict__ part, int f, int m, double (&v)[Q],
                                            double *__restrict__ tot)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (w < Q) {
        double s = 0.0;
        for (int q = lane; q < m; q += 64) s += part[(long long)(f + q) * Q + w];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
        if (lane == 0) tot[w] = s;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < Q; k++) v[k] = tot[k];
}

}  // namespace pgdev
