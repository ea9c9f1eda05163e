// pg_pairsum.hpp -- FP64 correlations of listed pairs by waves, MI355X (gfx950),
// shared by the construction (corr.hip) and the dense average (cormat.hip).
#pragma once

#include <hip/hip_runtime.h>

namespace pgdev {

// FP64 r of P pairs by one wave, exactly as the FP64 oracle forms it: the rounded products
// added in time order (lane p < P holds
// pair p in e and gets its unclamped sum).  The wave walks the pairs' rows TC
// time points at a time: TC / 2 lanes read one row's run of TC * 8 bytes, 16
// bytes each, so a load covers whole runs of a few rows (a thread per pair
// touches 64 rows per load and is bound by the texture addresser: 64 lines
// for 512 bytes).  The rounded products go through LDS and lane p adds pair
// p's in time order; the next run's loads are in flight under the sums.
// P * TC = 1024 keeps 16 loads of 16 bytes per lane in flight.  P = 64 sums
// on every lane (bulk); P = 16 takes t / 64 dependent rounds instead of t / 16
// (lists that do not fill the chip with 64 pairs per wave).
// Two layouts.  Rows: z[i * n + l], l = 0 .. len - 1; a row starts at a multiple
// of 8 bytes only (odd t): d2u has that alignment, and a global 16-byte load
// needs no more than 4; the run past t is read at the row's last two points
// and masked to zero (a zero product leaves the sum: it starts at +0); offsets
// below 2^32 and len >= 2, checked by the caller.  CHUNKS (P = 64): zchunk_copy's
// z[(c * n + i) * 16 + l % 16], zero past t, so every run is one 128-byte line
// (a row's run straddles two); c counts the chunks from the caller's first.
// prod: this wave's P * (TC + 2) doubles of LDS; the padding of two keeps the
// 16-byte row reads off each other's banks.
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));
typedef double d2a __attribute__((ext_vector_type(2)));
template <int P, bool CHUNKS = false>
struct PairSum {
    static constexpr int TC = 1024 / P, LPR = TC / 2, RPL = 64 / LPR, M = P / RPL, LDP = TC + 2;
    static constexpr int LDS_DOUBLES = P * LDP;
    static_assert(!CHUNKS || TC == 16, "a chunk is one run");
    // rows: n apart, len points each; chunks: len / 16 chunks of n rows
    static __device__ __forceinline__ double run(int2 e, const double *__restrict__ z, int n, int len, double sum,
                                                 int lane, double *__restrict__ prod)
    {
#pragma clang fp contract(off)
        const int rl = lane / LPR, cl = 2 * (lane % LPR);
        const unsigned stride = CHUNKS ? (unsigned)TC : (unsigned)n;
        unsigned oa[M], ob[M];
#pragma unroll
        for (int m = 0; m < M; m++) {
            oa[m] = (unsigned)__shfl(e.x, m * RPL + rl) * stride;
            ob[m] = (unsigned)__shfl(e.y, m * RPL + rl) * stride;
        }
        d2a x[M], y[M];
        auto load = [&](int l0) {
            if (CHUNKS) {
                const double *zc = z + (long long)l0 * n + cl;  // chunk l0 / 16
#pragma unroll
                for (int m = 0; m < M; m++) {
                    x[m] = *(const d2a *)(zc + oa[m]);
                    y[m] = *(const d2a *)(zc + ob[m]);
                }
            } else {
                const unsigned l = (unsigned)min(l0 + cl, len - 2);
#pragma unroll
                for (int m = 0; m < M; m++) {
                    x[m] = *(const d2u *)(z + (oa[m] + l));
                    y[m] = *(const d2u *)(z + (ob[m] + l));
                }
            }
        };
        load(0);
        for (int l0 = 0; l0 < len; l0 += TC) {
            const int l = l0 + cl;
            const bool both = CHUNKS || l + 1 < len, last = !CHUNKS && l + 1 == len;  // last: point len - 1, read as .y
#pragma unroll
            for (int m = 0; m < M; m++) {
                const double p0 = x[m].x * y[m].x, p1 = x[m].y * y[m].y;
                d2a w;
                w.x = both ? p0 : (last ? p1 : 0.0);
                w.y = both ? p1 : 0.0;
                *(d2a *)(prod + (m * RPL + rl) * LDP + cl) = w;
            }
            __builtin_amdgcn_wave_barrier();
            if (l0 + TC < len) load(l0 + TC);
            if (P == 64 || lane < P) {
#pragma unroll
                for (int k = 0; k < TC; k += 2) {
                    const d2a w = *(const d2a *)(prod + lane * LDP + k);
                    sum += w.x;
                    sum += w.y;
                }
            }
            __builtin_amdgcn_wave_barrier();
        }
        return sum;
    }
};
constexpr int PAIR_LDS = PairSum<64>::LDS_DOUBLES > PairSum<16>::LDS_DOUBLES ? PairSum<64>::LDS_DOUBLES
                                                                             : PairSum<16>::LDS_DOUBLES;
static_assert(PAIR_LDS % 2 == 0, "each wave's products start 16-byte aligned");

__device__ __forceinline__ double clamp_r(double r) { return r > 1.0 ? 1.0 : (r < -1.0 ? -1.0 : r); }

}  // namespace pgdev
