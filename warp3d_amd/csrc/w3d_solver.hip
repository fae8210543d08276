// w3d_solver.hip -- device Jacobi-preconditioned conjugate gradients on the
// assembled stiffness (the upper-triangular VSS arrays expanded to a full
// symmetric CSR), FP64 throughout.
//
// Stands in for the reference's direct solve of the assembled equations
// (drive_assemble_solve.f:654 -> drive_pardiso.f:11, and the MKL iterative
// option of the same driver); the reference's element-by-element PCG
// (old_code/EBE_solver/lnpcg_ser/lnpcg.f) is the precedent for a Jacobi
// preconditioner.  Every reduction is a fixed tree (per-workgroup partial
// sums, then every workgroup over the partials), so a solve is bitwise
// repeatable.
#include <hip/hip_runtime.h>

#include <cmath>
#include <mutex>

#include "w3d_internal.h"

namespace w3d {

constexpr int kRedBlock = 256;

// Work memory of w3d_solve_pcg_static, which allocates nothing: the vectors
// of up to kStaticMaxEq equations, then the scalars, state and partial
// sums.  Each device holds its own copy for the life of the process;
// concurrent calls on one device share it.
constexpr int64_t kStaticWords =
    (int64_t)kPcgVectors * kStaticMaxEq + kPcgTail;
static __device__ __align__(256) double scratch[kStaticWords];

// The device address of this device's scratch (hipGetSymbolAddress once
// per device, with that device current; the host-side name is not a
// device address).
int solver_static_scratch(int device, double** out) {
  static std::mutex mu;
  static double* addr[kMaxDevices] = {};
  if (device < 0 || device >= kMaxDevices) return W3D_ERR_ARG;
  std::lock_guard<std::mutex> lk(mu);
  if (!addr[device]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p)
      return W3D_ERR_DEVICE;
    addr[device] = static_cast<double*>(p);
  }
  *out = addr[device];
  return W3D_OK;
}

// vals[k] = the assembled word vidx[k] (diagonal words first, then the
// upper-triangle coefficients): the full CSR values of an assembly
__global__ void k_csr_values(const double* __restrict__ diag,
                             const double* __restrict__ coef, int neq,
                             const uint32_t* __restrict__ vidx, int64_t nnz,
                             double* __restrict__ vals) {
  int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < nnz) {
    uint32_t v = vidx[k];
    vals[k] = v < (uint32_t)neq ? diag[v] : coef[v - neq];
  }
}

// ---------------------------------------------------------------------
// Products with the full CSR rows, one row group (the free equations of
// one structure node, which share their columns: up to three consecutive
// rows of one length) per kGrpLanes lanes.  A lane reads a column index and
// its vector entry once for the group's rows, so an entry of the matrix
// costs 9.3 bytes (8 + 4/3) and a third of a gather instead of 12 bytes
// and one, and the value streams of the rows are each contiguous.  32
// lanes: the 81 columns of a structured brick's node are three entries a
// lane, loaded together, and a 1,000-node system still spreads over 32,000
// lanes.  Bound by memory on large systems (124,740 equations, 9.5 M
// entries: 28 us, 4.7 TB/s).  Each row sums its lanes' strided shares in a
// fixed butterfly, so products are bitwise repeatable.  Workgroups of 256:
// of 512, an iteration on one to three systems of 2,000 to 3,600 equations
// took 7.3 to 7.8 us for 6.0 to 7.4.
// ---------------------------------------------------------------------
constexpr int kGrpLanes = 32;
constexpr int kMulBlock = 256;
constexpr int kGrpPerWg = kMulBlock / kGrpLanes;

// A lane's share of one row group: kGrpAhead entries of each row and the
// vector words of their columns (past the end: the group's last entry).
constexpr int kGrpAhead = 3;
template <typename W>
struct GrpTile {
  RowGroup d;
  int c[kGrpAhead];
  double a[3][kGrpAhead];
  W x[kGrpAhead];
};
template <typename W>
__device__ __forceinline__ void tile_columns(const RowGroups& A, int lane,
                                             int from, GrpTile<W>& t) {
  const int len = t.d.len();
  const int32_t* cp = A.col + t.d.k0;
#pragma unroll
  for (int u = 0; u < kGrpAhead; ++u) {
    const int k = from + lane + u * kGrpLanes;
    t.c[u] = cp[k < len ? k : len - 1];
  }
}
template <typename W>
__device__ __forceinline__ void tile_entries(const double* __restrict__ val,
                                             const W* __restrict__ x,
                                             int lane, int from,
                                             GrpTile<W>& t) {
  const int len = t.d.len(), nr = t.d.rows();
  const double* v = val + t.d.k0;
  const int o1 = nr > 1 ? len : 0, o2 = nr > 2 ? 2 * len : 0;
#pragma unroll
  for (int u = 0; u < kGrpAhead; ++u) {
    const int k = from + lane + u * kGrpLanes;
    const int kk = k < len ? k : len - 1;
    t.a[0][u] = v[kk];
    t.a[1][u] = v[o1 + kk];
    t.a[2][u] = v[o2 + kk];
  }
#pragma unroll
  for (int u = 0; u < kGrpAhead; ++u) t.x[u] = x[t.c[u]];
}
// the first entries of group g, loaded ahead of the scalars a product needs
template <typename W>
__device__ __forceinline__ void tile_load(const RowGroups& A,
                                          const double* __restrict__ val,
                                          const W* __restrict__ x, int g,
                                          int lane, GrpTile<W>& t) {
  t.d = A.grp[g];
  tile_columns(A, lane, 0, t);
  tile_entries(val, x, lane, 0, t);
}

// s[k] = row (row0 + k) . f(x) over the rows of the loaded group, every lane
// of the group holding the sums
template <typename W, typename F>
__device__ __forceinline__ void tile_product(const RowGroups& A,
                                             const double* __restrict__ val,
                                             const W* __restrict__ x,
                                             int lane, GrpTile<W>& t,
                                             const F& f, double (&s)[3]) {
  s[0] = s[1] = s[2] = 0.0;
  for (int from = 0;;) {
#pragma unroll
    for (int u = 0; u < kGrpAhead; ++u) {
      const double xv = f(t.x[u]);
      const bool in = from + lane + u * kGrpLanes < t.d.len();
#pragma unroll
      for (int k = 0; k < 3; ++k) s[k] = in ? s[k] + t.a[k][u] * xv : s[k];
    }
    from += kGrpAhead * kGrpLanes;
    if (from >= t.d.len()) break;
    tile_columns(A, lane, from, t);
    tile_entries(val, x, lane, from, t);
  }
#pragma unroll
  for (int off = kGrpLanes / 2; off >= 1; off >>= 1)
#pragma unroll
    for (int r = 0; r < 3; ++r) s[r] = s[r] + __shfl_xor(s[r], off, kGrpLanes);
}

// sums of N values over the workgroup of NT threads in a fixed order
// (butterfly in each wave, the waves in order); every thread gets them
template <int N, int NT>
__device__ __forceinline__ void block_sums(double (&v)[N],
                                           double (*s_red)[NT / 64]) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1)
#pragma unroll
    for (int k = 0; k < N; ++k) v[k] = v[k] + __shfl_xor(v[k], off);
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int k = 0; k < N; ++k) s_red[k][threadIdx.x >> 6] = v[k];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < N; ++k) {
    v[k] = s_red[k][0];
#pragma unroll
    for (int w = 1; w < NT / 64; ++w) v[k] = v[k] + s_red[k][w];
  }
  __syncthreads();
}

// y = A x
__global__ void __launch_bounds__(kMulBlock)
    k_grp_spmv(RowGroups A, const double* __restrict__ val,
               const double* __restrict__ x, double* __restrict__ y) {
  const int lane = threadIdx.x % kGrpLanes;
  const int g = blockIdx.x * kGrpPerWg + threadIdx.x / kGrpLanes;
  if (g >= A.ngrp) return;
  double s[3];
  GrpTile<double> t;
  tile_load(A, val, x, g, lane, t);
  tile_product(A, val, x, lane, t, [](double w) { return w; }, s);
  if (lane < t.d.rows())
    y[t.d.row0 + lane] = lane == 0 ? s[0] : lane == 1 ? s[1] : s[2];
}

// ---------------------------------------------------------------------
// Jacobi-PCG over one system or a batch of independent ones, one launch an
// iteration, in the form of the usual recurrences that needs one set of sums
// (Meurant 1984): with u = D^-1 r and s = A p
//   alpha = g / (p, s),  g = (r, u)
//   beta = (g - 2 alpha (s, u) + alpha^2 (s, D^-1 s)) / g
//   x += alpha p, r -= alpha s, p = D^-1 r + beta p
// The bracket is (r, u) of the new r, formed from sums the old vectors give,
// so that beta does not wait for them; the next alpha takes the new (r, u)
// as summed.  A launch forms the scalars from the last launch's partial sums,
// the new r and p at the columns it gathers (from the old r, p, s and
// 1 / diag, 32 bytes a column, kept in two buffers by the launch's parity),
// s = A p of its own rows and the five sums (with r.r, for the test).  The
// matrix, column and vector words of a workgroup's first tile are loaded
// before the scalars are known: neither needs the other.
//
// s is a product and alpha a quotient of sums taken directly: with
// w = A u as the product, s = w + beta s and alpha = g / ((w, u) - beta g /
// alpha-) (Chronopoulos and Gear 1989, three sums) the recurrence's rounding
// errors cost slender or nearly incompressible models 5 to 60 % more
// iterations and up to twice the true residual (bricks in a row of 200, to
// 1e-8: 8,200 to 8,600 iterations, 11,700 to 12,800 so).
//
// A launch is a chain of dependent loads and two workgroup sums on small
// systems, and the host reads the states behind the device, so an iteration
// costs no synchronisation.  Measured an iteration, against two launches
// (product, vector update): 10.5 -> 8.0 us on three systems of 2,000 to 3,600
// equations, 32.4 -> 28.2 us (4.7 TB/s) on 124,740; with three sums 7.4 and
// 27.4, the request of three served models the same within 1 %.  Three waves
// a SIMD: at four, the next group's words (below) spilled, and a solve of
// 124,740 equations took 41 us an iteration.
// Each system's reductions run over its own workgroups in a
// fixed order, whose number depends on the system's size alone, so a
// system's iterates do not depend on the batch.  Every workgroup of a system
// reaches the same end-of-solve decision from the same partials and the
// first one writes it.  What other lanes read is never written by the same
// launch: the gathered rows, the partial sums and the gates are double, read
// at the launch's parity and written at the other, and state (done,
// iterations per system) is the host's.  x is updated in place, each entry
// by the one lane that reads it.
// ---------------------------------------------------------------------
template <bool BATCH>
__global__ void __launch_bounds__(kMulBlock)
    k_pcg_init(const PcgSys one, const PcgSys* __restrict__ sys,
               const int32_t* __restrict__ owner) {
  __shared__ double s_red[1][kMulBlock / 64];
  const int si =
      BATCH ? __builtin_amdgcn_readfirstlane(owner[blockIdx.x]) : 0;
  const PcgSys& S = BATCH ? sys[si] : one;
  const int wg = blockIdx.x - S.wg0;
  double v[1] = {0.0};  // b.b
  for (int i = wg * kMulBlock + threadIdx.x; i < S.n;
       i += S.nwg * kMulBlock) {
    const double bi = S.b[i];
    double ri = bi;
    if (S.single)
      ri = bi - S.ax()[i];
    else
      S.x[i] = 0.0;
    PcgRow q;
    q.r = ri;
    q.p = q.s = 0.0;
    q.rd = 1.0 / S.diag[i];
    S.row[1][i] = q;
    v[0] = v[0] + bi * bi;
  }
  block_sums<1, kMulBlock>(v, s_red);
  if (threadIdx.x == 0) S.part[S.off_bb() + wg] = v[0];
}

// one workgroup per system: |b|; a zero right-hand side is solved
template <bool BATCH>
__global__ void __launch_bounds__(kRedBlock)
    k_pcg_init2(const PcgSys one, const PcgSys* __restrict__ sys,
                int32_t* __restrict__ state, int32_t* __restrict__ gate,
                double* __restrict__ sc) {
  __shared__ double s_red[1][kRedBlock / 64];
  const PcgSys& S = BATCH ? sys[blockIdx.x] : one;
  double v[1] = {0.0};
  for (int i = threadIdx.x; i < S.nwg; i += kRedBlock)
    v[0] = v[0] + S.part[S.off_bb() + i];
  block_sums<1, kRedBlock>(v, s_red);
  if (threadIdx.x == 0) {
    sc[2 * blockIdx.x] = sqrt(v[0]);
    sc[2 * blockIdx.x + 1] = v[0];
    const int32_t end = v[0] == 0.0 ? (S.single ? kPcgZeroRhs : 1) : 0;
    state[2 * blockIdx.x] = end;
    state[2 * blockIdx.x + 1] = 0;
    gate[2 * blockIdx.x] = gate[2 * blockIdx.x + 1] = end;
  }
}

template <bool BATCH>
__global__ void __launch_bounds__(kMulBlock)
    __attribute__((amdgpu_waves_per_eu(3)))
    k_pcg_iter(const PcgSys one, const PcgSys* __restrict__ sys,
               const int32_t* __restrict__ owner, int it,
               int32_t* __restrict__ state, int32_t* __restrict__ gate,
               double* __restrict__ sc) {
  __shared__ double s_red[kPcgSums][kMulBlock / 64];
  const int si =
      BATCH ? __builtin_amdgcn_readfirstlane(owner[blockIdx.x]) : 0;
  const PcgSys& S = BATCH ? sys[si] : one;
  const int wg = blockIdx.x - S.wg0, par = it & 1;
  const int tid = threadIdx.x, lane = tid % kGrpLanes;
  if (gate[2 * si + par]) {
    if (wg == 0 && tid == 0) gate[2 * si + (par ^ 1)] = 1;
    return;
  }
  const PcgRow* __restrict__ row = S.row[par];
  int g = wg * kGrpPerWg + tid / kGrpLanes;
  GrpTile<PcgRow> t;
  PcgRow o;          // lane k < rows: row k's own vectors
  double xo;
  auto load = [&]() {  // of the group whose word and columns t has
    tile_entries(S.val, row, lane, 0, t);
    const int i = t.d.row0 + (lane < t.d.rows() ? lane : 0);
    o = row[i];
    xo = S.x[i];
  };
  if (g < S.A.ngrp) {
    t.d = S.A.grp[g];
    tile_columns(S.A, lane, 0, t);
    load();
  }
  double alpha = 0.0, beta = 0.0;
  if (it >= 0) {
    const double* pt = S.part + S.off_sums(par);
    double v[kPcgSums] = {};  // r.r, r.u, p.s, s.u, s.(s / diag)
    for (int i = tid; i < S.nwg; i += kMulBlock)
#pragma unroll
      for (int k = 0; k < kPcgSums; ++k) v[k] = v[k] + pt[k * S.nwg + i];
    block_sums<kPcgSums, kMulBlock>(v, s_red);
    // the end of the solve: |r| <= rtol |b| or the iteration limit (a batch
    // tests neither before its first iteration; a single solve also stops
    // on a residual that is no number)
    const double nr_ = sqrt(v[0]);
    const bool conv = nr_ <= S.rtol * sc[2 * si];
    if ((it > 0 || S.single) &&
        (conv || it >= S.maxit || (S.single && isnan(nr_)))) {
      if (wg == 0 && tid == 0) {
        state[2 * si] = conv ? 1 : 2;
        state[2 * si + 1] = it;
        gate[2 * si + (par ^ 1)] = 1;
        sc[2 * si + 1] = v[0];
      }
      return;
    }
    alpha = v[1] / v[2];
    beta = (v[1] + alpha * (alpha * v[4] - 2.0 * v[3])) / v[1];
  }
  // the new residual and direction of a row from its old vectors
  auto residual = [&](const PcgRow& q) { return q.r - alpha * q.s; };
  auto direction = [&](const PcgRow& q, double r) {
    return r * q.rd + beta * q.p;
  };
  double v[kPcgSums] = {};
  while (g < S.A.ngrp) {
    // the next group's word and columns come in behind this one's products
    const int gn = g + S.nwg * kGrpPerWg;
    GrpTile<PcgRow> nx;
    nx.d = S.A.grp[gn < S.A.ngrp ? gn : g];
    tile_columns(S.A, lane, 0, nx);
    const int i = t.d.row0 + lane;
    const bool own = lane < t.d.rows();
    PcgRow n;
    if (own) {
      n.rd = o.rd;
      n.r = residual(o);
      n.p = direction(o, n.r);
      if (it >= 0) S.x[i] = xo + alpha * o.p;
    }
    double y[3];
    tile_product(S.A, S.val, row, lane, t,
                 [&](const PcgRow& q) { return direction(q, residual(q)); },
                 y);
    if (own) {
      n.s = lane == 0 ? y[0] : lane == 1 ? y[1] : y[2];
      S.row[par ^ 1][i] = n;
      const double u = n.r * n.rd;
      v[0] = v[0] + n.r * n.r;
      v[1] = v[1] + n.r * u;
      v[2] = v[2] + n.p * n.s;
      v[3] = v[3] + n.s * u;
      v[4] = v[4] + n.s * (n.s * n.rd);
    }
    g = gn;
    if (g < S.A.ngrp) {
      t.d = nx.d;
#pragma unroll
      for (int u = 0; u < kGrpAhead; ++u) t.c[u] = nx.c[u];
      load();
    }
  }
  block_sums<kPcgSums, kMulBlock>(v, s_red);
  if (tid == 0)
#pragma unroll
    for (int k = 0; k < kPcgSums; ++k)
      S.part[S.off_sums(par ^ 1) + k * S.nwg + wg] = v[k];
}

// Workgroups of one system's launches: a tile of groups (rows) each up to
// the cap, then equal shares.  The caps bound the partial sums that every
// workgroup of the next launch reads again, and keep a launch's workgroups
// resident together at three waves a SIMD (124,740 equations: 28.1 us an
// iteration on 743; 27.4 and, on 867, 34.1 before the five sums).
int pcg_mul_wgs(int ngrp) {
  const int t = (ngrp + kGrpPerWg - 1) / kGrpPerWg;
  if (t < 1) return 1;
  const int per = (t + kPcgMaxMul - 1) / kPcgMaxMul;
  return (t + per - 1) / per;
}
int pcg_vec_wgs(int n) {
  const int t = (n + kRedBlock - 1) / kRedBlock;
  return t < 1 ? 1 : t > kPcgMaxVec ? kPcgMaxVec : t;
}

// state: 2 nsys words, the gates behind them
int launch_pcg_init(const PcgSys& one, hipStream_t s, int32_t* state,
                    double* sc) {
  hipLaunchKernelGGL(k_pcg_init<false>, dim3(one.nwg), dim3(kMulBlock), 0, s,
                     one, nullptr, nullptr);
  hipLaunchKernelGGL(k_pcg_init2<false>, dim3(1), dim3(kRedBlock), 0, s, one,
                     nullptr, state, state + 2, sc);
  return launch_pcg_iter(one, -1, state, sc, s);
}

int launch_pcg_iter(const PcgSys& one, int it, int32_t* state, double* sc,
                    hipStream_t s) {
  hipLaunchKernelGGL(k_pcg_iter<false>, dim3(one.nwg), dim3(kMulBlock), 0, s,
                     one, nullptr, nullptr, it, state, state + 2, sc);
  return hipGetLastError() == hipSuccess ? W3D_OK : W3D_ERR_DEVICE;
}

int launch_pcg_batch_init(const PcgBatch& b, int32_t* state, double* sc,
                          hipStream_t s) {
  if (b.nsys <= 0) return W3D_OK;
  hipLaunchKernelGGL(k_pcg_init<true>, dim3(b.nwg), dim3(kMulBlock), 0, s,
                     PcgSys{}, b.sys, b.owner);
  hipLaunchKernelGGL(k_pcg_init2<true>, dim3(b.nsys), dim3(kRedBlock), 0, s,
                     PcgSys{}, b.sys, state, state + 2 * b.nsys, sc);
  return launch_pcg_batch_iter(b, -1, state, sc, s);
}

int launch_pcg_batch_iter(const PcgBatch& b, int it, int32_t* state,
                          double* sc, hipStream_t s) {
  if (b.nsys <= 0) return W3D_OK;
  hipLaunchKernelGGL(k_pcg_iter<true>, dim3(b.nwg), dim3(kMulBlock), 0, s,
                     PcgSys{}, b.sys, b.owner, it, state, state + 2 * b.nsys,
                     sc);
  return hipGetLastError() == hipSuccess ? W3D_OK : W3D_ERR_DEVICE;
}

// ---------------------------------------------------------------------
// Jacobi-preconditioned BiCGStab (van der Vorst 1992, right
// preconditioning) on the full CSR rows, FP64, three launches an iteration:
//   k_bicg_v   the test and beta, p = r + beta (p - omega v) at the
//              gathered columns (pairs (r / diag, (p - omega v) / diag)),
//              v = A D^-1 p, partial (rh, v)
//   k_bicg_t   alpha, s = r - alpha v at the gathered columns (pairs
//              (r / diag, v / diag)), t = A D^-1 s, partial (t, s), (t, t)
//   k_bicg_x   omega, x, r, the pairs of the next iteration, partial
//              (rh, r), (r, r)
// (9,360 equations: 113 us an iteration with a launch per operation and a
// host read, 20 us so.)
// As in the PCG above every workgroup forms the scalars from the partial
// sums of the launches before (a fixed order: a solve is bitwise
// repeatable) and the first one writes them to sc for later launches:
// [0], [1] rho by iteration parity, [2] alpha, [3] omega, [4] (r, r),
// [5] |b|.  gate[0..2] close the three launches; none reads a gate that it
// writes.  A breakdown (a zero rho, (rh, v) or last omega) ends the solve
// with x at the last iterate.
// ---------------------------------------------------------------------
constexpr int kBicgScalars = 8;
enum { kBicgConv = 1, kBicgLimit = 2, kBicgBreak = 3, kBicgZero = 4,
       kBicgNan = 5 };

struct BicgSys {
  RowGroups A;
  const double* val;
  const double* b;
  double *x, *r, *rh, *p, *v, *s, *t, *dinv;
  double2 *rp2;             // (r, p - omega v) / diag
  double2 *rv2;             // (r, v) / diag
  double *part;             // rv nmul, ts nmul, tt nmul, rho nvec, rr nvec
  double *sc;
  int32_t* state;           // done, iterations; then the gates
  int32_t* gate;
  double rtol;
  int32_t n, nmul, nvec, maxit;
};

__global__ void __launch_bounds__(kRedBlock) k_bicg_init(const BicgSys S) {
  __shared__ double s_red[1][kRedBlock / 64];
  double v[1] = {0.0};
  for (int i = blockIdx.x * kRedBlock + threadIdx.x; i < S.n;
       i += S.nvec * kRedBlock) {
    // dinv holds the row's diagonal (0 when the pattern has none)
    const double d = S.dinv[i], di = d != 0.0 ? 1.0 / d : 1.0;
    const double bi = S.b[i];
    S.dinv[i] = di;
    S.x[i] = 0.0;
    S.r[i] = bi;
    S.rh[i] = bi;
    S.rp2[i] = make_double2(bi * di, 0.0);
    S.p[i] = 0.0;
    S.v[i] = 0.0;
    v[0] = v[0] + bi * bi;
  }
  block_sums<1, kRedBlock>(v, s_red);
  if (threadIdx.x == 0) {  // rh = r = b: rho and (r, r) are (b, b)
    S.part[3 * S.nmul + blockIdx.x] = v[0];
    S.part[3 * S.nmul + S.nvec + blockIdx.x] = v[0];
  }
}

__global__ void __launch_bounds__(kRedBlock) k_bicg_init2(const BicgSys S) {
  __shared__ double s_red[1][kRedBlock / 64];
  double v[1] = {0.0};
  for (int i = threadIdx.x; i < S.nvec; i += kRedBlock)
    v[0] = v[0] + S.part[3 * S.nmul + i];
  block_sums<1, kRedBlock>(v, s_red);
  if (threadIdx.x == 0) {
    for (int k = 0; k < kBicgScalars; ++k) S.sc[k] = 0.0;
    S.sc[4] = v[0];
    S.sc[5] = sqrt(v[0]);
    const int32_t end = sqrt(v[0]) == 0.0 ? kBicgZero : 0;
    S.state[0] = end;
    S.state[1] = 0;
    S.gate[0] = S.gate[1] = S.gate[2] = end;
  }
}

// the diagonal of every row (0 when absent)
__global__ void __launch_bounds__(kMulBlock)
    k_grp_diag(RowGroups A, const double* __restrict__ val,
               double* __restrict__ diag) {
  const int lane = threadIdx.x % kGrpLanes;
  const int g = blockIdx.x * kGrpPerWg + threadIdx.x / kGrpLanes;
  if (g >= A.ngrp) return;
  const RowGroup gd = A.grp[g];
  const int row0 = gd.row0, nr = gd.rows(), len = gd.len();
  const int64_t k0 = gd.k0;
  double d[3] = {0.0, 0.0, 0.0};
  for (int k = lane; k < len; k += kGrpLanes) {
    const int j = A.col[k0 + k] - row0;
    if (j == 0) d[0] = val[k0 + k];
    if (j == 1 && nr > 1) d[1] = val[k0 + len + k];
    if (j == 2 && nr > 2) d[2] = val[k0 + 2 * (int64_t)len + k];
  }
#pragma unroll
  for (int off = kGrpLanes / 2; off >= 1; off >>= 1)
#pragma unroll
    for (int r = 0; r < 3; ++r) d[r] = d[r] + __shfl_xor(d[r], off, kGrpLanes);
  if (lane < nr) diag[row0 + lane] = lane == 0 ? d[0] : lane == 1 ? d[1] : d[2];
}

__global__ void __launch_bounds__(kMulBlock)
    __attribute__((amdgpu_waves_per_eu(4)))
    k_bicg_v(const BicgSys S, int it) {
  __shared__ double s_red[2][kMulBlock / 64];
  if (S.gate[0]) return;
  const int wg = blockIdx.x, tid = threadIdx.x, lane = tid % kGrpLanes;
  const double2* __restrict__ w2 = S.rp2;
  int g = wg * kGrpPerWg + tid / kGrpLanes;
  GrpTile<double2> t;
  if (g < S.A.ngrp) tile_load(S.A, S.val, w2, g, lane, t);
  double v[2] = {0.0, 0.0};  // rho, (r, r)
  for (int i = tid; i < S.nvec; i += kMulBlock) {
    v[0] = v[0] + S.part[3 * S.nmul + i];
    v[1] = v[1] + S.part[3 * S.nmul + S.nvec + i];
  }
  block_sums<2, kMulBlock>(v, s_red);
  const double rho = v[0], rho1 = S.sc[(it - 1) & 1], alpha1 = S.sc[2],
               omega1 = S.sc[3];
  int end = 0;
  if (it > 0) {  // the residual of iteration it
    if (!isfinite(v[1]))
      end = kBicgNan;
    else if (sqrt(v[1]) / S.sc[5] <= S.rtol)
      end = kBicgConv;
    else if (it >= S.maxit)
      end = kBicgLimit;
  }
  if (!end && (rho == 0.0 || (it > 0 && (rho1 == 0.0 || omega1 == 0.0))))
    end = kBicgBreak;
  if (wg == 0 && tid == 0) {
    S.sc[4] = v[1];
    S.sc[it & 1] = rho;
    if (end) {
      S.state[0] = end;
      S.state[1] = it;
      S.gate[1] = S.gate[2] = 1;
    }
  }
  if (end) return;
  const double beta = it > 0 ? (rho / rho1) * (alpha1 / omega1) : 0.0;
  double dot[1] = {0.0};
  while (g < S.A.ngrp) {
    double s[3];
    tile_product(S.A, S.val, w2, lane, t,
                 [&](const double2& w) { return w.x + beta * w.y; }, s);
    if (lane < t.d.rows()) {
      const int i = t.d.row0 + lane;
      const double ri = S.r[i], di = S.dinv[i];
      const double vi = lane == 0 ? s[0] : lane == 1 ? s[1] : s[2];
      // p, v: the last iteration's on entry, this one's on exit
      S.p[i] = ri + beta * (S.p[i] - omega1 * S.v[i]);
      S.v[i] = vi;
      S.rv2[i] = make_double2(ri * di, vi * di);
      dot[0] = dot[0] + S.rh[i] * vi;
    }
    g += S.nmul * kGrpPerWg;
    if (g < S.A.ngrp) tile_load(S.A, S.val, w2, g, lane, t);
  }
  double d2[1] = {dot[0]};
  block_sums<1, kMulBlock>(d2, s_red);
  if (tid == 0) S.part[wg] = d2[0];
}

__global__ void __launch_bounds__(kMulBlock)
    k_bicg_t(const BicgSys S, int it) {
  __shared__ double s_red[2][kMulBlock / 64];
  if (S.gate[1]) return;
  const int wg = blockIdx.x, tid = threadIdx.x, lane = tid % kGrpLanes;
  const double2* __restrict__ w2 = S.rv2;
  int g = wg * kGrpPerWg + tid / kGrpLanes;
  GrpTile<double2> t;
  if (g < S.A.ngrp) tile_load(S.A, S.val, w2, g, lane, t);
  double rv[1] = {0.0};
  for (int i = tid; i < S.nmul; i += kMulBlock) rv[0] = rv[0] + S.part[i];
  block_sums<1, kMulBlock>(rv, s_red);
  if (rv[0] == 0.0) {
    if (wg == 0 && tid == 0) {
      S.state[0] = kBicgBreak;
      S.state[1] = it;
      S.gate[2] = 1;
    }
    return;
  }
  const double alpha = S.sc[it & 1] / rv[0];
  if (wg == 0 && tid == 0) S.sc[2] = alpha;
  double v[2] = {0.0, 0.0};  // (t, s), (t, t)
  while (g < S.A.ngrp) {
    double s[3];
    tile_product(S.A, S.val, w2, lane, t,
                 [&](const double2& w) { return w.x - alpha * w.y; }, s);
    if (lane < t.d.rows()) {
      const int i = t.d.row0 + lane;
      const double ti = lane == 0 ? s[0] : lane == 1 ? s[1] : s[2];
      const double si = S.r[i] - alpha * S.v[i];
      S.s[i] = si;
      S.t[i] = ti;
      v[0] = v[0] + ti * si;
      v[1] = v[1] + ti * ti;
    }
    g += S.nmul * kGrpPerWg;
    if (g < S.A.ngrp) tile_load(S.A, S.val, w2, g, lane, t);
  }
  block_sums<2, kMulBlock>(v, s_red);
  if (tid == 0) {
    S.part[S.nmul + wg] = v[0];
    S.part[2 * S.nmul + wg] = v[1];
  }
}

__global__ void __launch_bounds__(kRedBlock) k_bicg_x(const BicgSys S) {
  __shared__ double s_red[2][kRedBlock / 64];
  const int wg = blockIdx.x;
  if (S.gate[2]) {
    if (wg == 0 && threadIdx.x == 0) S.gate[0] = S.gate[1] = 1;
    return;
  }
  double v[2] = {0.0, 0.0};
  for (int i = threadIdx.x; i < S.nmul; i += kRedBlock) {
    v[0] = v[0] + S.part[S.nmul + i];
    v[1] = v[1] + S.part[2 * S.nmul + i];
  }
  block_sums<2, kRedBlock>(v, s_red);
  // (t, t) = 0: s is already the residual of x (a converged half step)
  const double omega = v[1] != 0.0 ? v[0] / v[1] : 0.0, alpha = S.sc[2];
  if (wg == 0 && threadIdx.x == 0) S.sc[3] = omega;
  v[0] = v[1] = 0.0;  // (rh, r), (r, r)
  for (int i = wg * kRedBlock + threadIdx.x; i < S.n;
       i += S.nvec * kRedBlock) {
    const double di = S.dinv[i], pi = S.p[i], si = S.s[i];
    const double y = pi * di, z = si * di;
    S.x[i] = (S.x[i] + alpha * y) + omega * z;
    const double ri = si - omega * S.t[i];
    S.r[i] = ri;
    S.rp2[i] = make_double2(ri * di, (pi - omega * S.v[i]) * di);
    v[0] = v[0] + S.rh[i] * ri;
    v[1] = v[1] + ri * ri;
  }
  block_sums<2, kRedBlock>(v, s_red);
  if (threadIdx.x == 0) {
    S.part[3 * S.nmul + wg] = v[0];
    S.part[3 * S.nmul + S.nvec + wg] = v[1];
  }
}

int bicgstab_words(int n, int ngrp) {
  return 11 * n + kBicgScalars + 4 + 3 * pcg_mul_wgs(ngrp) +
         2 * pcg_vec_wgs(n);
}

int bicgstab(int n, const RowGroups& A, const double* val, const double* b,
             double* x, double* work, double rtol, int maxit, int* iters,
             double* relres, int32_t* const h[2], const hipEvent_t ev[2],
             hipStream_t st) {
  BicgSys S{};
  S.A = A;
  S.val = val;
  S.b = b;
  S.x = x;
  S.rp2 = reinterpret_cast<double2*>(work);  // work: 16-byte aligned
  S.rv2 = S.rp2 + n;
  S.r = reinterpret_cast<double*>(S.rv2 + n);
  S.rh = S.r + n;
  S.p = S.rh + n;
  S.v = S.p + n;
  S.s = S.v + n;
  S.t = S.s + n;
  S.dinv = S.t + n;
  S.sc = S.dinv + n;
  S.state = reinterpret_cast<int32_t*>(S.sc + kBicgScalars);
  S.gate = S.state + 2;
  S.part = S.sc + kBicgScalars + 4;
  S.rtol = rtol;
  S.n = n;
  S.nmul = pcg_mul_wgs(A.ngrp);
  S.nvec = pcg_vec_wgs(n);
  S.maxit = maxit;
  const dim3 gm(S.nmul), tm(kMulBlock), gv(S.nvec), tv(kRedBlock);
  if (A.ngrp > 0)
    hipLaunchKernelGGL(k_grp_diag, dim3((A.ngrp + kGrpPerWg - 1) / kGrpPerWg),
                       tm, 0, st, A, val, S.dinv);
  hipLaunchKernelGGL(k_bicg_init, gv, tv, 0, st, S);
  hipLaunchKernelGGL(k_bicg_init2, dim3(1), tv, 0, st, S);
  const int32_t* state = nullptr;
  const int rc = solve_poll(
      [&](int it) {
        hipLaunchKernelGGL(k_bicg_v, gm, tm, 0, st, S, it);
        if (it < maxit) {
          hipLaunchKernelGGL(k_bicg_t, gm, tm, 0, st, S, it);
          hipLaunchKernelGGL(k_bicg_x, gv, tv, 0, st, S);
        }
        return hipGetLastError() == hipSuccess ? W3D_OK : W3D_ERR_DEVICE;
      },
      1, maxit, kPollChunk, kPollChunk, S.state, h, ev, st, &state);
  if (rc) return rc;
  const int end = state[0];
  *iters = state[1];
  *relres = 0.0;
  if (end == kBicgZero) return W3D_OK;
  double v[2];
  if (hipMemcpyAsync(v, S.sc + 4, sizeof v, hipMemcpyDeviceToHost, st) !=
          hipSuccess ||
      hipStreamSynchronize(st) != hipSuccess)
    return W3D_ERR_DEVICE;
  *relres = std::sqrt(v[0]) / v[1];
  return end == kBicgConv ? W3D_OK : W3D_ERR_NUMERIC;
}

// the system owning global tile t (tile0 ascending, system 0 at tile 0)
template <typename S>
__device__ __forceinline__ int owner(const S* __restrict__ sys, int nsys,
                                     int t) {
  int lo = 0, hi = nsys - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (sys[mid].tile0 <= t)
      lo = mid;
    else
      hi = mid - 1;
  }
  return __builtin_amdgcn_readfirstlane(lo);
}

// sum of v over the workgroup (256 threads), the same order every time;
// every thread gets the result
__device__ __forceinline__ double block_sum(double v, double* s_red) {
  s_red[threadIdx.x] = v;
  __syncthreads();
  for (int w = kRedBlock / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
      s_red[threadIdx.x] = s_red[threadIdx.x] + s_red[threadIdx.x + w];
    __syncthreads();
  }
  const double r = s_red[0];
  __syncthreads();
  return r;
}

// sum of n partials (strided per thread, then the tree)
__device__ __forceinline__ double sum_partials(const double* __restrict__ v,
                                               int n, double* s_red) {
  double t = 0.0;
  for (int i = threadIdx.x; i < n; i += kRedBlock) t = t + v[i];
  return block_sum(t, s_red);
}

// ---------------------------------------------------------------------
// Batched Newton bookkeeping (one tile = kTileRows equations and
// kTileRows constrained dofs of one problem)
// ---------------------------------------------------------------------
__global__ void __launch_bounds__(kRedBlock)
    k_residual_batch(const ResSys* __restrict__ sys, int nsys,
                     double* __restrict__ part) {
  __shared__ double s_red[kRedBlock];
  const int si = owner(sys, nsys, blockIdx.x);
  const ResSys& S = sys[si];
  const int t = blockIdx.x - S.tile0;
  const int k = t * kTileRows + threadIdx.x;
  double res = 0.0, rea = 0.0, load = 0.0;
  if (threadIdx.x < kTileRows) {
    if (k < S.neq) {
      const double v = -S.ifv[S.eqdof[k]];
      S.rhs[k] = v;
      res = v * v;
    }
    if (k < S.ncdof) {
      const double v = S.ifv[S.cdof[k]];
      rea = v * v;
    }
    if (k < S.nldof) load = S.ifv[S.ldof[k]];
  }
  res = block_sum(res, s_red);
  rea = block_sum(rea, s_red);
  load = block_sum(load, s_red);
  if (threadIdx.x == 0) {
    double* P = part + 3 * (int64_t)S.tile0;
    P[t] = res;
    P[S.ntile + t] = rea;
    P[2 * S.ntile + t] = load;
  }
}

__global__ void __launch_bounds__(kRedBlock)
    k_residual_sums(const ResSys* __restrict__ sys,
                    const double* __restrict__ part, double* __restrict__ out) {
  __shared__ double s_red[kRedBlock];
  const ResSys& S = sys[blockIdx.x];
  const double* P = part + 3 * (int64_t)S.tile0;
  const double res = sum_partials(P, S.ntile, s_red);
  const double rea = sum_partials(P + S.ntile, S.ntile, s_red);
  const double load = sum_partials(P + 2 * S.ntile, S.ntile, s_red);
  if (threadIdx.x == 0) {
    double* o = out + 8 * (int64_t)blockIdx.x;
    o[0] = res;
    o[1] = rea;
    o[2] = load;
    for (int f = 0; f < 4; ++f) o[3 + f] = (double)S.flags[f];
    o[7] = 0.0;
  }
}

__global__ void __launch_bounds__(kRedBlock)
    k_du_batch(const ResSys* __restrict__ sys, int nsys) {
  const int si = owner(sys, nsys, blockIdx.x);
  const ResSys& S = sys[si];
  if (!S.solve) return;
  const int t = blockIdx.x - S.tile0;
  const int k = t * kTileRows + threadIdx.x;
  if (threadIdx.x < kTileRows && k < S.neq) {
    const int d = S.eqdof[k];
    S.du[d] = S.du[d] + S.x[k];
  }
}

__global__ void k_axpy1(int64_t n, double* __restrict__ u,
                        const double* __restrict__ du) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) u[i] = u[i] + du[i];
}

__global__ void k_start_increment(const int32_t* __restrict__ eqdof, int neq,
                                  const int32_t* __restrict__ cdof,
                                  const double* __restrict__ cimp, int ncdof,
                                  double sf, double disp,
                                  double* __restrict__ du) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < neq) {
    const int d = eqdof[k];
    du[d] = sf * du[d];
  }
  if (k < ncdof) du[cdof[k]] = disp * cimp[k];
}

int launch_start_increment(const int32_t* eqdof, int neq, const int32_t* cdof,
                           const double* cimp, int ncdof, double sf,
                           double disp, double* du, hipStream_t s) {
  const int n = neq > ncdof ? neq : ncdof;
  if (n > 0)
    hipLaunchKernelGGL(k_start_increment, dim3((n + 255) / 256), dim3(256), 0,
                       s, eqdof, neq, cdof, cimp, ncdof, sf, disp, du);
  return hipGetLastError() == hipSuccess ? W3D_OK : W3D_ERR_DEVICE;
}

int launch_residual_batch(const ResSys* d_sys, int nsys, int ntile_total,
                          double* part, double* out, hipStream_t s) {
  if (nsys <= 0) return W3D_OK;
  if (ntile_total > 0)
    hipLaunchKernelGGL(k_residual_batch, dim3(ntile_total), dim3(kRedBlock),
                       0, s, d_sys, nsys, part);
  hipLaunchKernelGGL(k_residual_sums, dim3(nsys), dim3(kRedBlock), 0, s,
                     d_sys, part, out);
  return hipGetLastError() == hipSuccess ? W3D_OK : W3D_ERR_DEVICE;
}

int launch_du_batch(const ResSys* d_sys, int nsys, int ntile_total,
                    hipStream_t s) {
  if (nsys <= 0 || ntile_total <= 0) return W3D_OK;
  hipLaunchKernelGGL(k_du_batch, dim3(ntile_total), dim3(kRedBlock), 0, s,
                     d_sys, nsys);
  return hipGetLastError() == hipSuccess ? W3D_OK : W3D_ERR_DEVICE;
}

int launch_axpy1(int64_t n, double* u, const double* du, hipStream_t s) {
  if (n > 0)
    hipLaunchKernelGGL(k_axpy1, dim3((unsigned)((n + 255) / 256)), dim3(256),
                       0, s, n, u, du);
  return hipGetLastError() == hipSuccess ? W3D_OK : W3D_ERR_DEVICE;
}

namespace {
inline unsigned nblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }
}

int solver_csr_values(const double* diag, const double* coef, int neq,
                      const uint32_t* vidx, int64_t nnz, double* vals,
                      hipStream_t s) {
  if (nnz > 0)
    hipLaunchKernelGGL(k_csr_values, dim3(nblk(nnz, 256)), dim3(256), 0, s,
                       diag, coef, neq, vidx, nnz, vals);
  return hipGetLastError() == hipSuccess ? W3D_OK : W3D_ERR_DEVICE;
}

int solver_spmv(const RowGroups& A, const double* val, const double* x,
                double* y, hipStream_t s) {
  if (A.ngrp > 0)
    hipLaunchKernelGGL(k_grp_spmv, dim3(nblk(A.ngrp, kGrpPerWg)),
                       dim3(kMulBlock), 0, s, A, val, x, y);
  return hipGetLastError() == hipSuccess ? W3D_OK : W3D_ERR_DEVICE;
}

}  // namespace w3d
