// w3d_wave.h -- the lanes of a wave: ordering of their LDS traffic, exchanges
// between the four lanes of a quad.
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

template <int CTRL>
__device__ inline int qperm(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ inline double qperm(double v) {
  return __hiloint2double(qperm<CTRL>(__double2hiint(v)),
                          qperm<CTRL>(__double2loint(v)));
}
// the quad's exchanges: with the neighbour (1 0 3 2), across (2 3 0 1)
constexpr int kDppNext = 0xB1, kDppCross = 0x4E;
// the quad's sum, the same bits in its four lanes (its lanes branch on such
// sums together): without contraction, as an addend that is a product would
// otherwise go into a multiply-add whose two sides the lanes round unlike
template <typename T>
__device__ inline T qsum(T v) {
#pragma clang fp contract(off)
  v = v + qperm<kDppNext>(v);
  return v + qperm<kDppCross>(v);
}
// the value of the quad's lane S
template <int S, typename T>
__device__ inline T qbcast(T v) {
  return qperm<S * 0x55>(v);
}
// the argument of the lane's own number
__device__ inline double qpick(int sub, double a, double b, double c,
                               double d) {
  const double lo = sub & 1 ? b : a, hi = sub & 1 ? d : c;
  return sub & 2 ? hi : lo;
}

}  // namespace w3d
