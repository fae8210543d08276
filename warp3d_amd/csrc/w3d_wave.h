// w3d_wave.h -- ordering of a wave's own LDS traffic.
#pragma once

#include <hip/hip_runtime.h>

namespace w3d {

// Wave-level synchronisation: the lanes of one wave exchange data through
// their own LDS slab, so the wave only has to order its own LDS traffic.  The
// barrier alone keeps instructions from being scheduled across it; the fences
// order the memory, whatever types the two sides access it by.  They cost no
// instruction: a wave's LDS accesses complete in order.
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

}  // namespace w3d
