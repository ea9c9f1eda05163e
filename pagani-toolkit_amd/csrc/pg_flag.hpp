// pg_flag.hpp -- a device flag that many waves raise, MI355X (gfx950).
#pragma once

#include <hip/hip_runtime.h>

namespace pgdev {

// *f = 1, *f being 0 or 1 and read by later launches only.  Every wave of a BFS
// level that found something raises the level's flag: counting the waves
// instead queues up to 180,000 atomics on one address, about 10 ns each.  The
// load keeps all but the first stores away.
__device__ __forceinline__ void raise(unsigned *f)
{
    if (__hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) == 0u)
        __hip_atomic_store(f, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace pgdev
