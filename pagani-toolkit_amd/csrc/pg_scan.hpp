// pg_scan.hpp -- exclusive scan of a short int array by one work-group,
// shared by the CSR builders of the dense average and the rewiring.  gfx950
// only.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>

namespace pgdev {

// out[q] = scale * (in[0] + ... + in[q - 1]) for q = 0 .. n (out[n] is the
// scaled total).  One work-group of 1024 threads: a contiguous run per wave,
// read 64 entries at a time (eight loads in flight), summed, and read again
// for the scan (58,000 entries: 57 us; 105 us with a run per thread).
__device__ __forceinline__ void block_scan_1024(const int *__restrict__ in, long long n, long long *__restrict__ out,
                                                long long scale)
{
    __shared__ long long wsum[17];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const long long per = (n + 1023) / 1024 * 64;
    const long long a = std::min<long long>(n, w * per), b = std::min<long long>(n, a + per);
    long long s = 0;
    for (long long q = a + lane; q < b; q += 512) {
        int v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = q + 64 * u < b ? in[q + 64 * u] : 0;
#pragma unroll
        for (int u = 0; u < 8; u++) s += v[u];
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (lane == 0) wsum[w] = s;
    __syncthreads();
    long long run = 0;
    for (int q = 0; q < w; q++) run += wsum[q];
    for (long long q0 = a; q0 < b; q0 += 512) {
        int v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = q0 + 64 * u + lane < b ? in[q0 + 64 * u + lane] : 0;
#pragma unroll
        for (int u = 0; u < 8; u++) {
            long long x = v[u];
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const long long y = __shfl_up(x, o);
                if (lane >= o) x += y;
            }
            if (q0 + 64 * u + lane < b) out[q0 + 64 * u + lane] = scale * (run + x - v[u]);
            run += __shfl(x, 63);
        }
    }
    if (w == 15 && lane == 0) out[n] = scale * run;
}

}  // namespace pgdev
