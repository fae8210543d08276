// w3d_mm10.hip -- gfx950 kernel of the mm10 crystal-plasticity update
// (Voce hardening, 12 fcc or bcc slip systems), four lanes per Gauss point.
//
// Reference routines restated (file:line under the reference's src/):
//   rstgp1.f:4327 drive_10_update ([R n+1] of the polar decomposition for
//   finite strains, R = I for small strains; the iteration-0 "extrapolate
//   off" linear-elastic update), mm10_a.f:29 mm10 (crystal
//   loop, averages, store), :480 mm10_init_cc_hist0, :1777/:1808/:2605
//   step-1 history initialisation, :2493 mm10_copy_cc_hist, :1689
//   mm10_setup_np1, :852 mm10_setup, :2086 mm10_setup_voche, :1102
//   mm10_solve_crystal, :2657 mm10_solve_strup (sub-stepping), :2901
//   mm10_solve (predictor :3032, corrector :3224), :664 mm10_tangent,
//   :3991 symmetrisation, :3375 mm10_update_rotation, :3447 expmw3x3,
//   :3493 mm10_output, :1195 mm10_update_euler_angles, :998
//   mm10_store_cryhist; mm10_b.f:63 formR2, :177 formJ11, :281 formJ12,
//   :377 formJ21, :439 formJ22, :1073 formR1, :1169 form_dbarp, :1239
//   form_wbarp, :1312 form_wp, :1513 symsw, :1613 iw, :1813 slipinc,
//   :1845 rs, :1896-2074 the Voce functions (with ehard's extra
//   sign(slip) factor on its rate term, :1978-1983, kept as written).
//
// Every array of the local problem has compile-time indices, so the whole
// solve stays in registers; the pivoting of the small eliminations is done
// with selects instead of indexed row swaps.  Operation order follows the
// reference, except that sums over the slip systems run as three systems a
// lane and two exchanges in the quad, that C (D - dbar) is C D less the
// systems' C ms, and that each system's resolved shear and its power are
// formed once per residual or Jacobian and reused.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "w3d_internal.h"
#include "w3d_wave.h"

namespace w3d {
namespace {

// Four lanes (a quad) share a point: lane `sub` of the quad owns the slip
// systems 3 sub .. 3 sub + 2 and, of a matrix, the columns sub, sub + 4 (and
// sub + 8).  Sums over the systems are a partial sum of the lane's three and
// two exchanges inside the quad, which leave the same bits in all four
// lanes, so a quad's lanes always branch together.
constexpr int NSL = 3;            // systems of a lane
constexpr int kLanes = 64;
constexpr int kPts = kLanes / 4;  // points of a wave

struct Props {
  const CrystalDev* cr;
  double rate_n, tau_y, tau_v, voce_m, theta_0, iD_v, eps_dot_0_y;
  double atol, atol1, rtol, rtol1;
  int miter, alter_mode, angle_type;
};

// A lane's part of crystal_state (the Voce subset).  The slip tensors
// (mm10_setup's ms, qc) depend only on the plastic rotation at n and R n+1,
// so every sub-step shares one copy: ms and qc of the lane's systems, and
// their products C ms, which every residual and Jacobian takes (in LDS, word
// w of lane t at cms[w * kLanes + t]), and sigma_n + C D of the increment (LDS
// too, word w of point t at trial[w * kPts + t]).
struct CState {
  double* trial;
  double tt_rate, tinc, dg;
  double ms[NSL][6];
  double q[NSL][3];
  const double* cms;
  int sub;
  __device__ double cm(int j, int r) const { return cms[(6 * j + r) * kLanes]; }
};

// a value that is the same in every lane, in scalar registers
__device__ inline int uniform(int v) {
  return __builtin_amdgcn_readfirstlane(v);
}
__device__ inline double uniform(double v) {
  return __hiloint2double(uniform(__double2hiint(v)),
                          uniform(__double2loint(v)));
}
__device__ inline int64_t uniform(int64_t v) {
  return (int64_t)(uint32_t)uniform((int)v) |
         (int64_t)uniform((int)(v >> 32)) << 32;
}

__device__ inline double sgn(double x) { return x >= 0.0 ? 1.0 : -1.0; }

// x^y of the Voce functions: by repeated squaring when y is a whole number
// in [0, 127] (the rate and Voce exponents of practice, e.g. n = 20, m = 1
// or 5: some ulps from the correctly rounded power, far inside the local
// solve's tolerances), ocml's pow otherwise.  y is a material constant, so
// the branch is uniform.  Over an array, in place: the exponent's bits are
// tested once for all N values (uniform branches around straight runs of N
// products).
template <int N>
__device__ inline void vpow_arr(double* v, double y) {
  const int k = (int)y;
  if ((double)k == y && k >= 0 && k < 128) {
    double r[N];
#pragma unroll
    for (int j = 0; j < N; ++j) r[j] = 1.0;
#pragma unroll
    for (int i = 0; i < 7; ++i) {
      if (k >> i & 1) {
#pragma unroll
        for (int j = 0; j < N; ++j) r[j] = r[j] * v[j];
      }
      if ((k >> i) > 1) {
#pragma unroll
        for (int j = 0; j < N; ++j) v[j] = v[j] * v[j];
      }
    }
#pragma unroll
    for (int j = 0; j < N; ++j) v[j] = r[j];
  } else {
#pragma unroll
    for (int j = 0; j < N; ++j) v[j] = pow(v[j], y);
  }
}
__device__ inline double vpow(double x, double y) {
  vpow_arr<1>(&x, y);
  return x;
}

// [b] c with b 3x3 column-major
__device__ inline void mv3(double* a, const double* b, const double* c) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
    a[i] = b[i] * c[0] + b[i + 3] * c[1] + b[i + 6] * c[2];
}

// mm10_rt2rve of rt (3x3 column-major) -> rv (6x6 column-major)
__device__ inline void rt2rve(const double* rt, double* rv) {
#define RT(i, j) rt[((i)-1) + 3 * ((j)-1)]
#define RV(i, j) rv[((i)-1) + 6 * ((j)-1)]
  RV(1, 1) = RT(1, 1) * RT(1, 1);
  RV(1, 2) = RT(1, 2) * RT(1, 2);
  RV(1, 3) = RT(1, 3) * RT(1, 3);
  RV(1, 4) = 2.0 * RT(1, 1) * RT(1, 2);
  RV(1, 5) = 2.0 * RT(1, 3) * RT(1, 2);
  RV(1, 6) = 2.0 * RT(1, 1) * RT(1, 3);
  RV(2, 1) = RT(2, 1) * RT(2, 1);
  RV(2, 2) = RT(2, 2) * RT(2, 2);
  RV(2, 3) = RT(2, 3) * RT(2, 3);
  RV(2, 4) = 2.0 * RT(2, 1) * RT(2, 2);
  RV(2, 5) = 2.0 * RT(2, 3) * RT(2, 2);
  RV(2, 6) = 2.0 * RT(2, 1) * RT(2, 3);
  RV(3, 1) = RT(3, 1) * RT(3, 1);
  RV(3, 2) = RT(3, 2) * RT(3, 2);
  RV(3, 3) = RT(3, 3) * RT(3, 3);
  RV(3, 4) = 2.0 * RT(3, 1) * RT(3, 2);
  RV(3, 5) = 2.0 * RT(3, 3) * RT(3, 2);
  RV(3, 6) = 2.0 * RT(3, 1) * RT(3, 3);
  RV(4, 1) = RT(1, 1) * RT(2, 1);
  RV(4, 2) = RT(1, 2) * RT(2, 2);
  RV(4, 3) = RT(1, 3) * RT(2, 3);
  RV(4, 4) = RT(1, 1) * RT(2, 2) + RT(2, 1) * RT(1, 2);
  RV(4, 5) = RT(1, 2) * RT(2, 3) + RT(1, 3) * RT(2, 2);
  RV(4, 6) = RT(1, 1) * RT(2, 3) + RT(1, 3) * RT(2, 1);
  RV(5, 1) = RT(2, 1) * RT(3, 1);
  RV(5, 2) = RT(3, 2) * RT(2, 2);
  RV(5, 3) = RT(2, 3) * RT(3, 3);
  RV(5, 4) = RT(2, 1) * RT(3, 2) + RT(2, 2) * RT(3, 1);
  RV(5, 5) = RT(2, 2) * RT(3, 3) + RT(3, 2) * RT(2, 3);
  RV(5, 6) = RT(2, 1) * RT(3, 3) + RT(2, 3) * RT(3, 1);
  RV(6, 1) = RT(1, 1) * RT(3, 1);
  RV(6, 2) = RT(1, 2) * RT(3, 2);
  RV(6, 3) = RT(1, 3) * RT(3, 3);
  RV(6, 4) = RT(1, 1) * RT(3, 2) + RT(1, 2) * RT(3, 1);
  RV(6, 5) = RT(1, 2) * RT(3, 3) + RT(1, 3) * RT(3, 2);
  RV(6, 6) = RT(1, 1) * RT(3, 3) + RT(3, 1) * RT(1, 3);
#undef RV
}

// mm10_rt2rvw
__device__ inline void rt2rvw(const double* rt, double* rv) {
#define RW(i, j) rv[((i)-1) + 3 * ((j)-1)]
  RW(1, 1) = RT(2, 2) * RT(3, 3) - RT(2, 3) * RT(3, 2);
  RW(1, 2) = RT(2, 1) * RT(3, 3) - RT(2, 3) * RT(3, 1);
  RW(1, 3) = RT(2, 1) * RT(3, 2) - RT(2, 2) * RT(3, 1);
  RW(2, 1) = RT(1, 2) * RT(3, 3) - RT(1, 3) * RT(3, 2);
  RW(2, 2) = RT(1, 1) * RT(3, 3) - RT(1, 3) * RT(3, 1);
  RW(2, 3) = RT(1, 1) * RT(3, 2) - RT(1, 2) * RT(3, 1);
  RW(3, 1) = RT(1, 2) * RT(2, 3) - RT(1, 3) * RT(2, 2);
  RW(3, 2) = RT(1, 1) * RT(2, 3) - RT(1, 3) * RT(2, 1);
  RW(3, 3) = RT(1, 1) * RT(2, 2) - RT(1, 2) * RT(2, 1);
#undef RW
#undef RT
}

// Gaussian elimination with partial pivoting (first largest |pivot|) of the
// N columns the quad holds (column c in lane c & 3, slot c >> 2), with the
// right-hand sides among the remaining slots.  A column's owner finds its
// pivot and multipliers and the quad takes them from it; entries below the
// diagonal of finished columns are left as they fall, nothing reads them.
// rp: the pivots' reciprocals.  The eliminations do not skip zero
// multipliers as LAPACK's loops do (a divergent branch that saves nothing;
// adding a zero product changes no value, signed zeros aside).
template <int N, int SLOTS, int J = 0>
__device__ inline void quad_eliminate(double (&A)[SLOTS][7], double (&rp)[N]) {
  if constexpr (J < N) {
    double* col = A[J >> 2];
    int p = J;
    double amax = fabs(col[J]);
#pragma unroll
    for (int i = J + 1; i < N; ++i) {
      const double v = fabs(col[i]);
      if (v > amax) {
        amax = v;
        p = i;
      }
    }
    p = qbcast<(J & 3)>(p);
#pragma unroll
    for (int i = J + 1; i < N; ++i) {
      const bool sw = i == p;
#pragma unroll
      for (int s = 0; s < SLOTS; ++s) {
        const double a = A[s][J], b = A[s][i];
        A[s][J] = sw ? b : a;
        A[s][i] = sw ? a : b;
      }
    }
    const double r = 1.0 / col[J];
    rp[J] = qbcast<(J & 3)>(r);
#pragma unroll
    for (int i = J + 1; i < N; ++i) {
      const double m = qbcast<(J & 3)>(col[i] * r);
#pragma unroll
      for (int s = 0; s < SLOTS; ++s) A[s][i] = A[s][i] - m * A[s][J];
    }
    quad_eliminate<N, SLOTS, J + 1>(A, rp);
  }
}

// Back substitution of NY right-hand sides of every lane against the
// eliminated columns.
template <int N, int SLOTS, int NY, int K = N - 1>
__device__ inline void quad_backsub(const double (&A)[SLOTS][7],
                                    const double (&rp)[N],
                                    double (&y)[NY][N]) {
  if constexpr (K >= 0) {
#pragma unroll
    for (int c = 0; c < NY; ++c) y[c][K] = y[c][K] * rp[K];
#pragma unroll
    for (int i = 0; i < K; ++i) {
      const double u = qbcast<(K & 3)>(A[K >> 2][i]);
#pragma unroll
      for (int c = 0; c < NY; ++c) y[c][i] = y[c][i] - y[c][K] * u;
    }
    quad_backsub<N, SLOTS, NY, K - 1>(A, rp, y);
  }
}

// A x = b, b the last column (lane 3, slot 1); x in all four lanes.
template <int N>
__device__ inline void quad_solve(double (&A)[2][7], double (&x)[N]) {
  double rp[N], y[1][N];
  quad_eliminate<N, 2>(A, rp);
#pragma unroll
  for (int i = 0; i < N; ++i) y[0][i] = qbcast<3>(A[1][i]);
  quad_backsub<N, 2, 1>(A, rp, y);
#pragma unroll
  for (int i = 0; i < N; ++i) x[i] = y[0][i];
}

// DPOSV('U', 6, 1) with the stiffness
__device__ inline void chol_solve6(const double* __restrict__ ain, double* b) {
  double a[36];
#pragma unroll
  for (int k = 0; k < 36; ++k) a[k] = ain[k];
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < j; ++k) s = s + a[k + 6 * j] * a[k + 6 * j];
    double ajj = sqrt(a[j + 6 * j] - s);
    a[j + 6 * j] = ajj;
#pragma unroll
    for (int c = j + 1; c < 6; ++c) {
      double t = 0.0;
#pragma unroll
      for (int k = 0; k < j; ++k) t = t + a[k + 6 * j] * a[k + 6 * c];
      a[j + 6 * c] = (a[j + 6 * c] - t) / ajj;
    }
  }
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    double t = b[j];
#pragma unroll
    for (int k = 0; k < j; ++k) t = t - a[k + 6 * j] * b[k];
    b[j] = t / a[j + 6 * j];
  }
#pragma unroll
  for (int j = 5; j >= 0; --j) {
    b[j] = b[j] / a[j + 6 * j];
#pragma unroll
    for (int i = 0; i < j; ++i) b[i] = b[i] - b[j] * a[i + 6 * j];
  }
}

// mm10_setup of an increment D over tinc: effective strain increment (k_0 =
// 0: no geometric hardening)
__device__ inline void setup(const Props& p, CState& s, const double* D,
                             double tinc) {
  const double twothirds = 2.0 / 3.0;
  double t1 = D[0] * D[0] + D[1] * D[1] + D[2] * D[2];
  double t2 = D[3] * D[3] + D[4] * D[4] + D[5] * D[5];
  s.tinc = tinc;
  s.dg = sqrt(twothirds * (t1 + 0.5 * t2));
  if (p.alter_mode) s.dg = p.eps_dot_0_y * tinc;
}

// the trial stress sigma_n + C D of the increment
__device__ inline void set_trial(const Props& p, CState& s, const double* D,
                                 const double* sn, int64_t stride) {
  const double* C = p.cr->C;
  double t[6];
#pragma unroll
  for (int i = 0; i < 6; ++i) t[i] = C[i] * D[0];
#pragma unroll
  for (int j = 1; j < 6; ++j)
#pragma unroll
    for (int i = 0; i < 6; ++i) t[i] = t[i] + C[i + 6 * j] * D[j];
  // (the quad's lanes hold the same values; each writes them)
#pragma unroll
  for (int i = 0; i < 6; ++i) s.trial[i * kPts] = sn[i * stride] + t[i];
}

// mm10_a_mult_type_1: a = b c (3x3 column-major), the reference's order
__device__ inline void mul33(double* a, const double* b, const double* c) {
#pragma unroll
  for (int j = 0; j < 3; ++j)
#pragma unroll
    for (int i = 0; i < 3; ++i)
      a[i + 3 * j] = b[i] * c[3 * j] + b[i + 3] * c[1 + 3 * j] +
                     b[i + 6] * c[2 + 3 * j];
}

// mm10_setup: the lane's slip tensors rotated by the plastic rotation at n,
// and their products with the stiffness.  The vectors kept in the state are
// qc, by RT2RVW(R Rp_n^T) (mm10_a.f:891-892); with small strains (rot null,
// R = I) R Rp_n^T is Rp_n^T exactly and qc equals qs.  rot: the point's
// [R n+1], column-major at rot[k * SG].
__device__ inline void slip_geometry(const Props& p, const double* Rpn,
                                     double* cms, CState& s,
                                     const double* rot, int64_t SG) {
  double tn[9], rw[9];
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) tn[i + 3 * j] = Rpn[j + 3 * i];
  if (rot) {
    double R[9], w[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) R[k] = rot[k * SG];
    mul33(w, R, tn);
    rt2rvw(w, rw);
  } else {
    rt2rvw(tn, rw);
  }
#pragma unroll
  for (int i = 0; i < NSL; ++i) mv3(s.q[i], rw, p.cr->qs[NSL * s.sub + i]);
  {
    double RE[36];
    rt2rve(tn, RE);
#pragma unroll
    for (int i = 0; i < NSL; ++i) {
      const double* m0 = p.cr->ms[NSL * s.sub + i];
#pragma unroll
      for (int r = 0; r < 6; ++r) s.ms[i][r] = RE[r] * m0[0];
#pragma unroll
      for (int j = 1; j < 6; ++j)
#pragma unroll
        for (int r = 0; r < 6; ++r)
          s.ms[i][r] = s.ms[i][r] + RE[r + 6 * j] * m0[j];
    }
  }
  const double* C = p.cr->C;
#pragma unroll
  for (int r = 0; r < 6; ++r) {
    double c[6];
#pragma unroll
    for (int j = 0; j < 6; ++j) c[j] = C[r + 6 * j];
#pragma unroll
    for (int i = 0; i < NSL; ++i) {
      double v = c[0] * s.ms[i][0];
#pragma unroll
      for (int j = 1; j < 6; ++j) v = v + c[j] * s.ms[i][j];
      cms[(6 * i + r) * kLanes] = v;
    }
  }
  s.cms = cms;
}

__device__ inline void symsw(const double* s, const double* w, double* sw) {
  sw[0] = s[3] * w[2] - s[5] * w[1];
  sw[1] = s[3] * w[2] - s[4] * w[0];
  sw[2] = s[5] * w[1] + s[4] * w[0];
  sw[3] = 0.5 * (w[2] * (s[0] - s[1]) + w[0] * s[5] - w[1] * s[4]);
  sw[4] = 0.5 * (w[0] * (s[1] - s[2]) + w[1] * s[3] + w[2] * s[5]);
  sw[5] = 0.5 * (w[1] * (s[0] - s[2]) + w[0] * s[3] - w[2] * s[4]);
}

// dg n |tau|^(n-1) / tau^n: times (|rs| / tau)^(n-1) the slip's derivative
// dg n |rs|^(n-1) / tau^n.  Its sign on the negative tau of a stray iterate
// is that of tau^n, and the power of a broken exponent has none.
__device__ inline double flow_scale(const Props& p, double dg, double itt) {
  double v = dg * p.rate_n * itt;
  if (itt < 0.0) {
    const int k = (int)p.rate_n;
    if ((double)k != p.rate_n)
      v = __builtin_nan("");
    else if (!(k & 1))
      v = -v;
  }
  return v;
}

// resolved shears, (|rs| / tau)^(n-1) and slip increments of the lane's
// systems at x (stress) and tau
__device__ inline void slips(const Props& p, const CState& s, const double* x,
                             double tt, double* rs, double* pw, double* gam) {
  // one reciprocal of tau for the quotients (a few ulps from the quotients
  // themselves, far inside the local solve's tolerances)
  const double itt = 1.0 / tt, dgt = s.dg * itt;
#pragma unroll
  for (int i = 0; i < NSL; ++i) {
    rs[i] = x[0] * s.ms[i][0] + x[1] * s.ms[i][1] + x[2] * s.ms[i][2] +
            x[3] * s.ms[i][3] + x[4] * s.ms[i][4] + x[5] * s.ms[i][5];
    pw[i] = fabs(rs[i] * itt);
  }
  vpow_arr<NSL>(pw, p.rate_n - 1.0);
#pragma unroll
  for (int i = 0; i < NSL; ++i) gam[i] = dgt * pw[i] * rs[i];
}

// form_wp: the spin of all systems, qc weighted by slip and diffusion
__device__ inline void form_w(const Props& p, const CState& s,
                              const double* rs, const double* gam, double* w) {
  w[0] = w[1] = w[2] = 0.0;
#pragma unroll
  for (int i = 0; i < NSL; ++i) {
    const double c = rs[i] * s.tinc * p.iD_v + gam[i];
#pragma unroll
    for (int k = 0; k < 3; ++k) w[k] = w[k] + c * s.q[i][k];
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) w[k] = qsum(w[k]);
}

// formR1 at x, from the lane's slips (rs, gam) there: x - sigma_n -
// C (D - dbar) + 2 sym(x) w, with C dbar summed from the systems' C ms
__device__ inline void formR1_slips(const Props& p, const CState& s,
                                    const double* x,
                                    const double* rs, const double* gam,
                                    double* R1) {
  double cd[6], wp[3], sw[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) cd[k] = 0.0;
#pragma unroll
  for (int i = 0; i < NSL; ++i) {
    const double c = rs[i] * s.tinc * p.iD_v + gam[i];
#pragma unroll
    for (int k = 0; k < 6; ++k) cd[k] = cd[k] + c * s.cm(i, k);
  }
  form_w(p, s, rs, gam, wp);
  symsw(x, wp, sw);
#pragma unroll
  for (int k = 0; k < 6; ++k)
    R1[k] = x[k] - (s.trial[k * kPts] - qsum(cd[k])) + 2.0 * sw[k];
}

// formR1 at x with tau tt
__device__ inline void formR1(const Props& p, const CState& s,
                              const double* x, double tt, double* R1) {
  double rs[NSL], pw[NSL], gam[NSL];
  slips(p, s, x, tt, rs, pw, gam);
  formR1_slips(p, s, x, rs, gam, R1);
}

// h_voche (tau_l = 0)
__device__ inline double h_voche(const Props& p, const double* gam, double tt,
                                 double tau_n) {
  double h = 0.0;
  double ht = 1.0 - (tt - p.tau_y) / p.tau_v + 0.0 / (tt - p.tau_y);
  double f = vpow(fabs(ht), p.voce_m) * sgn(ht);
#pragma unroll
  for (int i = 0; i < NSL; ++i) h = h + f * fabs(gam[i]);
  return tau_n + p.theta_0 * qsum(h);
}

// formR (7 residuals); records the hardening rate
__device__ inline void formR(const Props& p, CState& s, double tau_n,
                             const double* x, double* R) {
  double rs[NSL], pw[NSL], gam[NSL];
  slips(p, s, x, x[6], rs, pw, gam);
  formR1_slips(p, s, x, rs, gam, R);
  double h = h_voche(p, gam, x[6], tau_n);
  R[6] = x[6] - h;
  s.tt_rate = (h - tau_n) / s.tinc;
}

// row r of column c (both known at compile time) of mm10_iw(w) + I
template <int C>
__device__ inline void add_iw(const double* w, double* col) {
  if (C == 0) { col[3] = col[3] + w[2]; col[5] = col[5] + w[1]; }
  if (C == 1) { col[3] = col[3] - w[2]; col[4] = col[4] + w[0]; }
  if (C == 2) { col[4] = col[4] - w[0]; col[5] = col[5] - w[1]; }
  if (C == 3) {
    col[0] = col[0] + 2.0 * w[2]; col[1] = col[1] + 2.0 * w[2];
    col[4] = col[4] + w[1]; col[5] = col[5] + w[0];
  }
  if (C == 4) {
    col[1] = col[1] + -2.0 * w[0]; col[2] = col[2] + 2.0 * w[0];
    col[3] = col[3] + -w[1]; col[5] = col[5] + -w[2];
  }
  if (C == 5) {
    col[0] = col[0] + -2.0 * w[1]; col[2] = col[2] + 2.0 * w[1];
    col[3] = col[3] + w[0]; col[4] = col[4] + w[2];
  }
  col[C] = col[C] + 1.0;
}

// formJ11 (N = 6) or formJ (N = 7) at (x, tt): the quad's lanes get the
// columns they own (A[slot][row]), column by column, so that one column's
// sums are live at a time.  |rs|^(n-1) / tau^n and the slips come from the
// powers (|rs| / tau)^(n-1) of the residual's slips.
template <int N, int C = 0>
__device__ inline void jac_columns(const CState& s, const double (*wv)[6],
                                   const double* dgdt, const double* e,
                                   const double* wp, double sc,
                                   double (&A)[2][7]) {
  if constexpr (C < 6) {
    double col[7];
#pragma unroll
    for (int r = 0; r < 6; ++r) col[r] = 0.0;
    double et = 0.0;
#pragma unroll
    for (int i = 0; i < NSL; ++i) {
      const double t = dgdt[i] * s.ms[i][C];
#pragma unroll
      for (int r = 0; r < 6; ++r) col[r] = col[r] + wv[i][r] * t;
      if (N == 7) et = et + e[i] * s.ms[i][C];
    }
#pragma unroll
    for (int r = 0; r < 6; ++r) col[r] = qsum(col[r]);
    add_iw<C>(wp, col);
    if (N == 7) col[6] = -(sc * qsum(et));
    const bool own = s.sub == (C & 3);
#pragma unroll
    for (int r = 0; r < N; ++r)
      A[C >> 2][r] = own ? col[r] : A[C >> 2][r];
    jac_columns<N, C + 1>(s, wv, dgdt, e, wp, sc, A);
  }
}

template <int N>
__device__ inline void formJ(const Props& p, const CState& s, const double* x,
                             double tt, double (&A)[2][7]) {
  double rs[NSL], pw[NSL], gam[NSL], wv[NSL][6], dgdt[NSL], e[NSL], wp[3];
  slips(p, s, x, tt, rs, pw, gam);
  const double itt = 1.0 / tt, nd = flow_scale(p, s.dg, itt);
#pragma unroll
  for (int i = 0; i < NSL; ++i) {
    dgdt[i] = nd * pw[i] + s.tinc * p.iD_v;
    double st[6];
    symsw(x, s.q[i], st);
#pragma unroll
    for (int r = 0; r < 6; ++r) wv[i][r] = 2.0 * st[r] + s.cm(i, r);
  }
  form_w(p, s, rs, gam, wp);
  double sc = 0.0, hm = 0.0, ht = 0.0;
  if (N == 7) {
    ht = 1.0 - (tt - p.tau_y) / p.tau_v + 0.0 / (tt - p.tau_y);
    hm = vpow(fabs(ht), p.voce_m);
    sc = p.theta_0 * nd;
#pragma unroll
    for (int i = 0; i < NSL; ++i) e[i] = hm * sgn(ht) * sgn(rs[i]) * pw[i];
  }
#pragma unroll
  for (int r = 0; r < 7; ++r) A[0][r] = A[1][r] = 0.0;
  jac_columns<N>(s, wv, dgdt, e, wp, sc, A);
  if (N == 7) {
    // J12 and J22
    double col[7], etau = 0.0;
#pragma unroll
    for (int r = 0; r < 6; ++r) col[r] = 0.0;
    const double dty = tt - p.tau_y;
    const double iht = 1.0 / fabs(ht), ntt = p.rate_n * itt;
#pragma unroll
    for (int i = 0; i < NSL; ++i) {
      const double dgdh = -ntt * gam[i];
#pragma unroll
      for (int r = 0; r < 6; ++r) col[r] = col[r] + wv[i][r] * dgdh;
      etau = etau + (p.voce_m * (-1.0 / p.tau_v - 0.0 / (dty * dty)) *
                         (fabs(gam[i]) * iht) -
                     fabs(gam[i]) * ntt * sgn(ht) * sgn(gam[i])) *
                        hm;
    }
    const bool own = s.sub == 2;
#pragma unroll
    for (int r = 0; r < 6; ++r) {
      const double v = qsum(col[r]);
      A[1][r] = own ? v : A[1][r];
    }
    const double v = 1.0 - p.theta_0 * qsum(etau);
    A[1][6] = own ? v : A[1][6];
  }
}

// (unrolled, so that the arrays it is given stay in registers)
template <int N>
__device__ inline bool any_nan(const double* x) {
  bool b = false;
#pragma unroll
  for (int i = 0; i < N; ++i) b |= isnan(x[i]);
  return b;
}

__device__ inline double dot6(const double* a, const double* b) {
  return a[0] * b[0] + a[1] * b[1] + a[2] * b[2] + a[3] * b[3] + a[4] * b[4] +
         a[5] * b[5];
}

// dx . (J^T R) of the columns the quad holds, then J dx = -R in place
template <int N>
__device__ inline double newton_step(double (&A)[2][7], const double* R,
                                     int sub, double (&dx)[N]) {
  double wv[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    wv[k] = 0.0;
#pragma unroll
    for (int l = 0; l < N; ++l) wv[k] = wv[k] + A[k][l] * R[l];
  }
#pragma unroll
  for (int r = 0; r < N; ++r) A[1][r] = sub == 3 ? -R[r] : A[1][r];
  quad_solve<N>(A, dx);
  double d = qpick(sub, dx[0], dx[1], dx[2], dx[3]) * wv[0];
  d = d + qpick(sub, dx[4], dx[5], N == 7 ? dx[N - 1] : 0.0, 0.0) * wv[1];
  return qsum(d);
}

// mm10_solve: predictor (6x6 Newton at fixed extrapolated tau) then the
// 7x7 corrector; Jl (49 words of the point at stride kPts, LDS) receives the
// Jacobian of the last corrector iteration
__device__ __forceinline__ void solve(const Props& p, CState& s, const double* D,
                      double tau_n, double tt_rate_n, const double* Dn,
                      int64_t dn_stride,
                      double* stress, double* tt, bool& fail, double dtinc,
                      double* Jl) {
  const double c = 1.0e-4, red = 0.5;
  const int mls = 10, mmin = 1;
  double x[7], inR1;
#pragma unroll
  for (int k = 0; k < 6; ++k) x[k] = stress[k];
  x[6] = *tt;
  {  // predictor
    double x1[6], R1[6], d1[6], d2[6], t1, t2, dtrace;
#pragma unroll
    for (int k = 0; k < 6; ++k) x1[k] = x[k];
#pragma unroll
    for (int k = 0; k < 6; ++k) d1[k] = D[k];
    dtrace = (d1[0] + d1[1] + d1[2]) / 3.0;
    d1[0] = d1[0] - dtrace;
    d1[1] = d1[1] - dtrace;
    d1[2] = d1[2] - dtrace;
    t1 = d1[0] * d1[0] + d1[1] * d1[1] + d1[2] * d1[2];
    t2 = d1[3] * d1[3] + d1[4] * d1[4] + d1[5] * d1[5];
    if (t1 + t2 == 0.0) {
#pragma unroll
      for (int k = 0; k < 6; ++k) d1[k] = 0.0;
    } else {
#pragma unroll
      for (int k = 0; k < 6; ++k) d1[k] = d1[k] / sqrt(t1 + t2);
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) d2[k] = Dn ? Dn[k * dn_stride] : 0.0;
    dtrace = (d2[0] + d2[1] + d2[2]) / 3.0;
    d2[0] = d2[0] - dtrace;
    d2[1] = d2[1] - dtrace;
    d2[2] = d2[2] - dtrace;
    t1 = d2[0] * d2[0] + d2[1] * d2[1] + d2[2] * d2[2];
    t2 = d2[3] * d2[3] + d2[4] * d2[4] + d2[5] * d2[5];
    if (t1 + t2 == 0.0) {
#pragma unroll
      for (int k = 0; k < 6; ++k) d2[k] = 0.0;
    } else {
#pragma unroll
      for (int k = 0; k < 6; ++k) d2[k] = d2[k] / sqrt(t1 + t2);
    }
    t1 = d1[0] * d2[0] + d1[1] * d2[1] + d1[2] * d2[2];
    t2 = d1[3] * d2[3] + d1[4] * d2[4] + d1[5] * d2[5];
    double cos_ang = t1 + t2 > 0.0 ? t1 + t2 : 0.0;
    double x2 = x[6] + cos_ang * tt_rate_n * dtinc;
    formR1(p, s, x1, x2, R1);
    double nR1 = sqrt(R1[0] * R1[0] + R1[1] * R1[1] + R1[2] * R1[2] +
                      R1[3] * R1[3] + R1[4] * R1[4] + R1[5] * R1[5]);
    inR1 = nR1;
    bool ok = true;
    int iter = 0;
    while (nR1 > p.atol1 && nR1 / inR1 > p.rtol1) {
      double A[2][7], dx1[6];
      formJ<6>(p, s, x1, x2, A);
      double dotR1 = R1[0] * R1[0] + R1[1] * R1[1] + R1[2] * R1[2] +
                     R1[3] * R1[3] + R1[4] * R1[4] + R1[5] * R1[5];
      double ls1 = 0.5 * dotR1;
      double ls2 = c * newton_step<6>(A, R1, s.sub, dx1);
      double alpha = 1.0;
      int ls = 0;
      for (;;) {
        double nlsx = ls1 + ls2 * alpha, xn[6];
#pragma unroll
        for (int k = 0; k < 6; ++k) xn[k] = x1[k] + alpha * dx1[k];
        formR1(p, s, xn, x2, R1);
        dotR1 = R1[0] * R1[0] + R1[1] * R1[1] + R1[2] * R1[2] +
                R1[3] * R1[3] + R1[4] * R1[4] + R1[5] * R1[5];
        nR1 = sqrt(dotR1);
        double nRs = 0.5 * dotR1;
        if (nRs <= nlsx || ls > mls) {
#pragma unroll
          for (int k = 0; k < 6; ++k) x1[k] = xn[k];
          break;
        }
        alpha = red * alpha;
        ls = ls + 1;
      }
      iter = iter + 1;
      if (iter > p.miter || any_nan<6>(x1)) {
        fail = true;
        ok = false;
        break;
      }
    }
    if (ok) {
#pragma unroll
      for (int k = 0; k < 6; ++k) x[k] = x1[k];
      x[6] = x2;
    }
  }
  {  // corrector
    int iter = 0;
    double R[7];
    formR(p, s, tau_n, x, R);
    double dotR = 0.0;
#pragma unroll
    for (int k = 0; k < 7; ++k) dotR = dotR + R[k] * R[k];
    double nR = sqrt(dotR), inR = nR;
    if (inR == 0.0) inR = inR1;
    while ((nR > p.atol && nR / inR > p.rtol) || iter < mmin) {
      double A[2][7], dx[7];
      formJ<7>(p, s, x, x[6], A);
      // the tangent takes the last iteration's Jacobian: parked in LDS
      // instead of held in registers across the loop
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int r = 0; r < 7; ++r)
          if (s.sub + 4 * k < 7) Jl[(r + 7 * (s.sub + 4 * k)) * kPts] = A[k][r];
      dotR = 0.0;
#pragma unroll
      for (int k = 0; k < 7; ++k) dotR = dotR + R[k] * R[k];
      double ls1 = 0.5 * dotR;
      double ls2 = c * newton_step<7>(A, R, s.sub, dx);
      double alpha = 1.0;
      int ls = 0;
      for (;;) {
        double nlsx = ls1 + ls2 * alpha, xn[7];
#pragma unroll
        for (int k = 0; k < 7; ++k) xn[k] = x[k] + alpha * dx[k];
        formR(p, s, tau_n, xn, R);
        dotR = 0.0;
#pragma unroll
        for (int k = 0; k < 7; ++k) dotR = dotR + R[k] * R[k];
        nR = sqrt(dotR);
        double nRs = 0.5 * dotR;
        if (nRs <= nlsx || ls > mls) {
#pragma unroll
          for (int k = 0; k < 7; ++k) x[k] = xn[k];
          break;
        }
        alpha = red * alpha;
        ls = ls + 1;
      }
      iter = iter + 1;
      if (iter > p.miter || any_nan<7>(x)) {
        fail = true;
        break;
      }
    }
  }
#pragma unroll
  for (int k = 0; k < 6; ++k) stress[k] = x[k];
  *tt = x[6];
}

// mm10_update_euler_angles (Kocks): angles of g (Rp R^T); with small
// strains (rot null, R = I) Rp R^T is Rp exactly
__device__ inline void euler_angles(const Props& p, const double* Rp_in,
                                    double* eul, const double* rot,
                                    int64_t SG) {
  const double pi = 3.141592653589793, one_eighty = 180.0;
  const double* g = p.cr->g;
  double Rp[9];
  if (rot) {  // mm10_a_mult_type_3t: Rp R^T
    double R[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) R[k] = rot[k * SG];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j)
        Rp[i + 3 * j] = Rp_in[i] * R[j] + Rp_in[i + 3] * R[j + 3] +
                        Rp_in[i + 6] * R[j + 6];
  } else {
#pragma unroll
    for (int k = 0; k < 9; ++k) Rp[k] = Rp_in[k];
  }
  double full[9];
#pragma unroll
  for (int j = 0; j < 3; ++j)
#pragma unroll
    for (int i = 0; i < 3; ++i)
      full[i + 3 * j] = g[i] * Rp[0 + 3 * j] + g[i + 3] * Rp[1 + 3 * j] +
                        g[i + 6] * Rp[2 + 3 * j];
  double psiK = atan2(full[2 + 3 * 1], full[2 + 3 * 0]);
  if (psiK < 0.0) psiK = psiK + 2.0 * pi;
  double phiK = atan2(full[1 + 3 * 2], full[0 + 3 * 2]);
  if (phiK < 0.0) phiK = phiK + 2.0 * pi;
  double f33 = full[8] > 1.0 ? 1.0 : full[8];
  double thetaK = acos(f33);
  if (p.angle_type == 1) {
    eul[0] = one_eighty / pi * psiK;
    eul[1] = one_eighty / pi * thetaK;
    eul[2] = one_eighty / pi * phiK;
  } else {
    eul[0] = psiK;
    eul[1] = thetaK;
    eul[2] = phiK;
  }
}

}  // namespace

// ---------------------------------------------------------------------
// A quad of lanes per Gauss point of an mm10 block (all its crystals):
// points kPts part .. kPts part + kPts - 1 of the work item on one wave.
//
// Latency and issue bound in FP64 (some 50 kflop a point in short dependent
// runs).  With a lane a point the local problem's arrays (49 Jacobian words,
// 12 systems) overflowed the 512 registers of a wave into 2.8 KB of scratch
// a lane, whose reloads from the Infinity Cache every chain waited on at one
// wave a SIMD; split over four lanes they fit half the registers, so two
// waves share a SIMD, a wave runs the longest of 16 local solves instead of
// 64, and small models spread over four times the waves.  167,000 points of
// a mixed mesh: 1,636 -> 672 us (54 % of the vector issue); 1.9 million:
// 32.6 -> 10.3 ms (72 %).
// ---------------------------------------------------------------------
constexpr int kCmsWords = 6 * NSL * kLanes;  // LDS of a wave: C ms,
constexpr int kJacWords = 49 * kPts;         // the parked Jacobians,
constexpr int kTriWords = 6 * kPts;          // the trial stresses and the
                                             // last accepted ones
constexpr int kMemWords = kCmsWords + kJacWords + 2 * kTriWords;

__device__ __forceinline__ void mm10_item(const DevModel& M,
                                          const WorkItem wi, int part,
                                          int step, int iter0_off,
                                          double* s_mem) {
  // (values the compiler may not carry in from outside the item, or across
  // the local solves: addresses formed from them are formed where they are
  // used instead of held in registers)
  int lane = threadIdx.x;
  asm volatile("" : "+v"(lane));
  const int pt = lane >> 2;
  int sub = lane & 3;
  if (kPts * part + pt >= wi.count) return;
  // (the block's and material's words are loaded per lane: the compiler
  // cannot know that nothing written here aliases them)
  const BlockDesc* bp = M.blocks + uniform(wi.blk);
  struct {
    int64_t q_off, hist_off;
    int geonl;
  } bd = {uniform(bp->q_off), uniform(bp->hist_off), uniform(bp->geonl)};
  const CpDesc* mp = &M.mats[uniform(bp->mat)].cp;
  const int G = uniform(bp->ngp);
  const int64_t SG = (int64_t)uniform(bp->span) * G;
  const int64_t crys_off = uniform(bp->crys_off);
  const int64_t q = wi.first + kPts * part + pt;  // point inside the block
  const int elem = (int)(q / G);
  const int ncry = uniform(bp->ncry);
  // the point's place in its block's arrays
  int qo = (int)q;
  auto fresh = [&](const double* base) {
    int k = qo;
    asm volatile("" : "+v"(k));
    return base + k;
  };
  const double* hist_n = M.hist_n + bd.hist_off;
  const double* uddt = M.uddt + 6 * bd.q_off;
  const double* stress_n = M.stress_n + 9 * bd.q_off;
  // finite strains: [R n+1] of the point (the recovery's), else R = I
  const double* rot_b = bd.geonl ? M.rot_tmp + 9 * bd.q_off : nullptr;
  const double dt = M.dt;
  double* Jl = s_mem + kCmsWords + pt;

  Props p;
  p.rate_n = uniform(mp->rate_n);
  p.tau_y = uniform(mp->tau_y);
  p.tau_v = uniform(mp->tau_v);
  p.voce_m = uniform(mp->voce_m);
  p.theta_0 = uniform(mp->theta_0);
  p.iD_v = uniform(mp->iD_v);
  p.eps_dot_0_y = uniform(mp->eps_dot_0_y);
  p.atol = uniform(mp->atol);
  p.atol1 = uniform(mp->atol1);
  p.rtol = uniform(mp->rtol);
  p.rtol1 = uniform(mp->rtol1);
  p.miter = uniform(mp->miter);
  p.alter_mode = uniform(mp->alter_mode);
  p.angle_type = uniform(mp->angle_type);

  // words the quad holds alike are stored four at a time, a lane a word
  // (n < 4: the last ones)
  auto put = [&](double* w, int n, double a, double b, double c2, double d) {
    const double v = qpick(sub, a, b, c2, d);
    if (sub < n) w[sub * SG] = v;
  };
  // crystal sums of the tangent, the stresses and the slips accumulate in
  // their output words (history 1-36, stress n+1 1-6, history 76-87), read
  // back only by the lane that writes them
  double t_work = 0.0, p_work = 0.0, p_strain = 0.0;
  bool cut = false;

  for (int c = 0; c < ncry; ++c) {
    p.cr = M.crys + crys_off + (int64_t)elem * ncry + c;
    const int64_t cb = (int64_t)(87 + 71 * c) * SG;
    // n-state of the crystal (mm10_copy_cc_hist; at step 1 the
    // mm10_init_cc_hist0 values)
    double tau_n, tt_rate_n;
    const double* stress_c = step == 1 ? stress_n : hist_n + cb;
    CState np1;
    np1.sub = sub;
    np1.trial = s_mem + kCmsWords + kJacWords + pt;
    double* ostress = np1.trial + kTriWords;
    {
      const double* hn = fresh(hist_n);
      double Rpn[9];
      if (step == 1) {
#pragma unroll
        for (int k = 0; k < 9; ++k) Rpn[k] = (k % 4 == 0) ? 1.0 : 0.0;
        tau_n = p.tau_y + 1.0e-5;
      } else {
#pragma unroll
        for (int k = 0; k < 9; ++k) Rpn[k] = hn[cb + (9 + k) * SG];
        tau_n = hn[cb + 42 * SG];
      }
      // np1 (mm10_setup_np1 + mm10_setup)
      slip_geometry(p, Rpn, s_mem + lane, np1,
                    rot_b ? fresh(rot_b) : nullptr, SG);
      tt_rate_n = hn[cb + 58 * SG];
    }
    // (C is read again where it is used, not held from here on)
    asm volatile("" : "+v"(p.cr));
    // mm10_solve_strup
    double D[6], stress[6], tt = tau_n, ott = tau_n;
    {
      const double* ud = fresh(uddt);
      const double* sn = fresh(stress_c);
#pragma unroll
      for (int k = 0; k < 6; ++k) D[k] = ud[k * SG];
#pragma unroll
      for (int k = 0; k < 6; ++k) stress[k] = sn[k * SG];
    }
    np1.tt_rate = 0.0;
    setup(p, np1, D, dt);
    double temp1 = dot6(D, D);
    double temp2 = dot6(stress, stress);
    const bool no_load = temp2 == 0.0 && temp1 == 0.0;
    bool fail = false;
    double curr_tt_rate = 0.0;
    // word k of the crystal's tangent into the point's average (history
    // words 0-35, word sub + 4 i the lane's)
    auto store_tangent = [&](int k, double v) {
      double* hn1 = M.hist_n1 + bd.hist_off + qo;
      hn1[k * SG] = c == 0 ? v : hn1[k * SG] + v;
    };
    if (iter0_off || no_load) {
      const double* C = p.cr->C;
#pragma unroll
      for (int i = 0; i < 9; ++i) store_tangent(sub + 4 * i, C[sub + 4 * i]);
      if (!no_load) {
        double R1[6];
        set_trial(p, np1, D, fresh(stress_c), SG);
        formR1(p, np1, stress, tt, R1);
#pragma unroll
        for (int k = 0; k < 6; ++k) stress[k] = stress[k] - R1[k];
      }
    } else {
      // the sub-steps run on np1 itself, their increments scaled from
      // the point's full-step values in memory (ud, dt); np1's full-step
      // values are formed again after the loop, so that they are not held
      // across the local solves
      double frac = 0.0, sstep = 1.0;
      int cuts = 0;
#pragma unroll
      for (int k = 0; k < 6; ++k) ostress[k * kPts] = stress[k];
      while (frac < 1.0) {
        const double* ud = fresh(uddt);
#pragma unroll
        for (int k = 0; k < 6; ++k) D[k] = ud[k * SG] * (sstep + frac);
        np1.tt_rate = 0.0;
        setup(p, np1, D, dt * (sstep + frac));
        set_trial(p, np1, D, fresh(stress_c), SG);
        asm volatile("" : "+v"(p.cr));
        tt = tau_n;
        // (Dn, the n strain increment)
        solve(p, np1, D, tau_n, tt_rate_n,
              step == 1 ? nullptr : fresh(hist_n) + cb + 18 * SG, SG, stress,
              &tt, fail, dt * sstep, Jl);
        if (fail) {
#pragma unroll
          for (int k = 0; k < 6; ++k) stress[k] = ostress[k * kPts];
          tt = ott;
          sstep = sstep * 0.5;
          cuts = cuts + 1;
          if (cuts > 4) break;
          fail = false;
        } else {
#pragma unroll
          for (int k = 0; k < 6; ++k) ostress[k * kPts] = stress[k];
          ott = tt;
          frac = frac + sstep;
        }
      }
      if (fail || isnan(tt) || any_nan<6>(stress)) {
        cut = true;
        break;
      }
      curr_tt_rate = np1.tt_rate;
      const double* ud = fresh(uddt);
#pragma unroll
      for (int k = 0; k < 6; ++k) D[k] = ud[k * SG];
      setup(p, np1, D, dt);
    }
    np1.tt_rate = curr_tt_rate;
    asm volatile("" : "+v"(sub), "+v"(qo), "+v"(p.cr));
    // mm10_store_cryhist: each word is stored as soon as it is formed
    double* h1 = M.hist_n1 + bd.hist_off + cb + qo;
    double slip[NSL];
#pragma unroll
    for (int k = 0; k < NSL; ++k) slip[k] = 0.0;
    put(h1, 4, stress[0], stress[1], stress[2], stress[3]);
    put(h1 + 4 * SG, 2, stress[4], stress[5], 0.0, 0.0);
    put(h1 + 18 * SG, 4, D[0], D[1], D[2], D[3]);
    put(h1 + 22 * SG, 2, D[4], D[5], 0.0, 0.0);
    put(h1 + 42 * SG, 4, tt, 0.0, 0.0, 0.0);  // and user words 1-3,
    put(h1 + 46 * SG, 2, 0.0, 0.0, 0.0, 0.0);  // 4-5,
    put(h1 + 51 * SG, 2, 0.0, 0.0, 0.0, 0.0);  // 9-10
    put(h1 + 58 * SG, 1, np1.tt_rate, 0.0, 0.0, 0.0);
    if (iter0_off || no_load) {
#pragma unroll
      for (int k = 6; k < 18; k += 4) put(h1 + k * SG, 4, 0.0, 0.0, 0.0, 0.0);
      put(h1 + 24 * SG, 4, 0.0, 0.0, 0.0, 0.0);
      put(h1 + 28 * SG, 2, 0.0, 0.0, 0.0, 0.0);
      put(h1 + 48 * SG, 3, 0.0, 0.0, 0.0, 0.0);
      put(h1 + 53 * SG, 4, 0.0, 0.0, 0.0, 0.0);
      put(h1 + 57 * SG, 1, 0.0, 0.0, 0.0, 0.0);
#pragma unroll
      for (int k = 59; k < 71; k += 4) put(h1 + k * SG, 4, 0.0, 0.0, 0.0, 0.0);
    } else {
      // ---- mm10_tangent: T = (J11 - J12 J21 / J22)^-1 C, symmetrised
      // unless the assembly is asymmetric.  Twelve columns in the quad: the
      // six of J11 - J12 J21 / J22, then C's
      {
        const double* C = p.cr->C;
        double A[3][7], rp[6], y[2][6];
        wave_sync();
        const double rj = 1.0 / Jl[48 * kPts];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const int cc = sub + 4 * k;
          if (k == 0 || sub < 2) {
            const double t = -(Jl[(6 + 7 * cc) * kPts] * rj);
#pragma unroll
            for (int r = 0; r < 6; ++r)
              A[k][r] = Jl[(r + 7 * cc) * kPts] + t * Jl[(r + 42) * kPts];
          } else {
#pragma unroll
            for (int r = 0; r < 6; ++r) A[k][r] = C[r + 6 * (sub - 2)];
          }
        }
#pragma unroll
        for (int r = 0; r < 6; ++r) A[2][r] = C[r + 6 * (sub + 2)];
        quad_eliminate<6, 3>(A, rp);
#pragma unroll
        for (int r = 0; r < 6; ++r) {
          y[0][r] = A[1][r];
          y[1][r] = A[2][r];
        }
        quad_backsub<6, 3, 2>(A, rp, y);
        wave_sync();
        if (sub >= 2)
#pragma unroll
          for (int r = 0; r < 6; ++r) Jl[(r + 6 * (sub - 2)) * kPts] = y[0][r];
#pragma unroll
        for (int r = 0; r < 6; ++r) Jl[(r + 6 * (sub + 2)) * kPts] = y[1][r];
        wave_sync();
#pragma unroll
        for (int i = 0; i < 9; ++i) {
          const int k = sub + 4 * i;
          double v = Jl[k * kPts];
          // (kept as formed for asymmetric assembly, :1165)
          if (!M.asym) v = (v + Jl[(k / 6 + 6 * (k % 6)) * kPts]) * 0.5;
          store_tangent(k, v);
        }
        wave_sync();
      }
      // ---- slips at the converged state (np1: full-step dg)
      double rs[NSL], pw[NSL], gam[NSL], wp[3];
      slips(p, np1, stress, tt, rs, pw, gam);
      form_w(p, np1, rs, gam, wp);
      // ---- mm10_update_rotation: Rp = expm(W(wbarp)) Rp_n (Rp_n read
      // again here)
      {
        double Rpe[9], Rp1[9], eul[3];
        const double* hn = fresh(hist_n);
        const double* rot = rot_b ? fresh(rot_b) : nullptr;
#pragma unroll
        for (int k = 0; k < 9; ++k)
          Rpe[k] = step == 1 ? ((k % 4 == 0) ? 1.0 : 0.0)
                             : hn[cb + (9 + k) * SG];
        double wb[3] = {wp[0], wp[1], wp[2]};
        if (rot) {  // form_wbarp takes qs, of Rp_n alone
          double tn[9], rw[9], w0[3] = {0.0, 0.0, 0.0};
#pragma unroll
          for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) tn[i + 3 * j] = Rpe[j + 3 * i];
          rt2rvw(tn, rw);
#pragma unroll
          for (int i = 0; i < NSL; ++i) {
            const double cw = rs[i] * np1.tinc * p.iD_v + gam[i];
            double qi[3];
            mv3(qi, rw, p.cr->qs[NSL * sub + i]);
#pragma unroll
            for (int k = 0; k < 3; ++k) w0[k] = w0[k] + cw * qi[k];
          }
#pragma unroll
          for (int k = 0; k < 3; ++k) wb[k] = qsum(w0[k]);
        }
        double W[9] = {0.0, -wb[2], -wb[1], wb[2], 0.0, -wb[0],
                       wb[1], wb[0], 0.0};  // column-major of wv2wt
        double alpha = sqrt(W[1 + 3 * 2] * W[1 + 3 * 2] +
                            W[0 + 3 * 2] * W[0 + 3 * 2] +
                            W[0 + 3 * 1] * W[0 + 3 * 1]);
        double A[9];
        if (alpha < 1.0e-16) {
#pragma unroll
          for (int k = 0; k < 9; ++k) A[k] = 0.0;
        } else {
          double ca = (1.0 - cos(alpha)) / (alpha * alpha);
          double sa = sin(alpha) / alpha;
#pragma unroll
          for (int j = 0; j < 3; ++j) {
#pragma unroll
            for (int i = 0; i < 3; ++i) A[i + 3 * j] = sa * W[i + 3 * j];
#pragma unroll
            for (int l = 0; l < 3; ++l) {
              double t = ca * W[l + 3 * j];
#pragma unroll
              for (int i = 0; i < 3; ++i)
                A[i + 3 * j] = A[i + 3 * j] + t * W[i + 3 * l];
            }
          }
        }
        A[0] = A[0] + 1.0;
        A[4] = A[4] + 1.0;
        A[8] = A[8] + 1.0;
#pragma unroll
        for (int j = 0; j < 3; ++j)
#pragma unroll
          for (int i = 0; i < 3; ++i)
            Rp1[i + 3 * j] = A[i] * Rpe[0 + 3 * j] + A[i + 3] * Rpe[1 + 3 * j] +
                             A[i + 6] * Rpe[2 + 3 * j];
        euler_angles(p, Rp1, eul, rot, SG);
        put(h1 + 6 * SG, 4, eul[0], eul[1], eul[2], Rp1[0]);
        put(h1 + 10 * SG, 4, Rp1[1], Rp1[2], Rp1[3], Rp1[4]);
        put(h1 + 14 * SG, 4, Rp1[5], Rp1[6], Rp1[7], Rp1[8]);
      }
      // ---- mm10_output
      double dif[NSL], edt[6], dbarp[6], t1, t2;
#pragma unroll
      for (int k = 0; k < 6; ++k) edt[k] = dbarp[k] = 0.0;
#pragma unroll
      for (int i = 0; i < NSL; ++i) {
        dif[i] = rs[i] * np1.tinc * p.iD_v;
#pragma unroll
        for (int k = 0; k < 6; ++k) {
          edt[k] = edt[k] + dif[i] * np1.ms[i][k];
          dbarp[k] = dbarp[k] + gam[i] * np1.ms[i][k];
        }
      }
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        edt[k] = qsum(edt[k]);
        dbarp[k] = qsum(dbarp[k]);
      }
      put(h1 + 65 * SG, 4, edt[0] / np1.tinc, edt[1] / np1.tinc,
          edt[2] / np1.tinc, edt[3] / np1.tinc);
      put(h1 + 69 * SG, 2, edt[4] / np1.tinc, edt[5] / np1.tinc, 0.0, 0.0);
      t1 = edt[0] * edt[0] + edt[1] * edt[1] + edt[2] * edt[2];
      t2 = edt[3] * edt[3] + edt[4] * edt[4] + edt[5] * edt[5];
      double ed_dot = sqrt(2.0 / 3.0 * (t1 + 0.5 * t2));
      const double u14 = ed_dot / np1.tinc;
      t_work = t_work + dot6(stress, D);
      double ee[6];
#pragma unroll
      for (int k = 0; k < 6; ++k) ee[k] = stress[k];
      chol_solve6(p.cr->C, ee);
      if (rot_b) {  // ee = RT2RVE(R) C^-1 sigma (exact for R = I)
        const double* rot = fresh(rot_b);
        double R[9], er[36], t[6];
#pragma unroll
        for (int k = 0; k < 9; ++k) R[k] = rot[k * SG];
        rt2rve(R, er);
#pragma unroll
        for (int i = 0; i < 6; ++i) {
          double a = er[i] * ee[0];
#pragma unroll
          for (int j = 1; j < 6; ++j) a = a + er[i + 6 * j] * ee[j];
          t[i] = a;
        }
#pragma unroll
        for (int k = 0; k < 6; ++k) ee[k] = t[k];
      }
      put(h1 + 24 * SG, 4, ee[0], ee[1], ee[2], ee[3]);
      put(h1 + 28 * SG, 2, ee[4], ee[5], 0.0, 0.0);
      double ewwe[6], ep[6];
      symsw(ee, wp, ewwe);
#pragma unroll
      for (int k = 0; k < 6; ++k) ep[k] = dbarp[k] + ewwe[k];
      put(h1 + 59 * SG, 4, ep[0] / np1.tinc, ep[1] / np1.tinc,
          ep[2] / np1.tinc, ep[3] / np1.tinc);
      put(h1 + 63 * SG, 2, ep[4] / np1.tinc, ep[5] / np1.tinc, 0.0, 0.0);
      t1 = ep[0] * ep[0] + ep[1] * ep[1] + ep[2] * ep[2];
      t2 = ep[3] * ep[3] + ep[4] * ep[4] + ep[5] * ep[5];
      const double u10 = sqrt(2.0 / 3.0 * (t1 + 0.5 * t2)) / np1.tinc;
#pragma unroll
      for (int k = 0; k < 6; ++k) ep[k] = ep[k] + edt[k];
      t1 = ep[0] * ep[0] + ep[1] * ep[1] + ep[2] * ep[2];
      t2 = ep[3] * ep[3] + ep[4] * ep[4] + ep[5] * ep[5];
      const double p_strain_inc = sqrt(2.0 / 3.0 * (t1 + 0.5 * t2));
      p_strain = p_strain + p_strain_inc;
      p_work = p_work + dot6(stress, ep);
      double ec_dot = p_strain_inc / np1.tinc, n_eff;
      if (ec_dot > 0.0) {
#pragma unroll
        for (int k = 0; k < 6; ++k) ep[k] = ep[k] / np1.tinc;
        n_eff = 0.0;
        const double nd = flow_scale(p, np1.dg, 1.0 / tt);
#pragma unroll
        for (int i = 0; i < NSL; ++i) {
          double dgdt = nd * pw[i] + np1.tinc * p.iD_v;
          const double* m = np1.ms[i];
          double a = m[0] * ep[0] + m[1] * ep[1] + m[2] * ep[2];
          double b = m[3] * ep[3] + m[4] * ep[4] + m[5] * ep[5];
          double ec_slip = a + 0.5 * b;
          double q1 = rs[i] * dgdt / ec_dot;
          double q2 = ec_slip / ec_dot / np1.tinc;
          n_eff = n_eff + (2.0 / 3.0) * q1 * q2;
        }
        n_eff = qsum(n_eff);
      } else {
        n_eff = 1.0e10;
      }
      double s_tr = (stress[0] + stress[1] + stress[2]) / 3.0;
      double se0 = stress[0] - s_tr, se1 = stress[1] - s_tr,
             se2 = stress[2] - s_tr;
      t1 = se0 * se0 + se1 * se1 + se2 * se2;
      t2 = stress[3] * stress[3] + stress[4] * stress[4] +
           stress[5] * stress[5];
      s_tr = sqrt(1.5 * (t1 + 2.0 * t2));
      double B_eff;
      if (ec_dot < 1.0e-100)
        B_eff = 0.0;
      else if (n_eff > 100.0)
        B_eff = -1.0;
      else
        B_eff = ec_dot / pow(s_tr, n_eff);
      put(h1 + 53 * SG, 4, u10, n_eff, s_tr, B_eff);
      put(h1 + 57 * SG, 1, u14, 0.0, 0.0, 0.0);
#pragma unroll
      for (int i = 0; i < NSL; ++i) slip[i] = gam[i] + dif[i];
      // the first system of the largest slip, and the active systems
      double maxslip = 0.0;
      int sysID = 0;
#pragma unroll
      for (int i = 0; i < NSL; ++i) {
        double cs = fabs(slip[i]);
        if (cs > maxslip) {
          maxslip = cs;
          sysID = NSL * sub + i + 1;
        }
      }
      auto larger = [&](double om, int oid) {
        const bool t = om > maxslip || (om == maxslip && oid < sysID);
        maxslip = t ? om : maxslip;
        sysID = t ? oid : sysID;
      };
      larger(qperm<kDppNext>(maxslip), qperm<kDppNext>(sysID));
      larger(qperm<kDppCross>(maxslip), qperm<kDppCross>(sysID));
      const double rate = maxslip / np1.tinc;
      int numAct = 0;
      maxslip = 0.1 * maxslip;
#pragma unroll
      for (int i = 0; i < NSL; ++i)
        if (fabs(slip[i]) >= maxslip) numAct = numAct + 1;
      put(h1 + 48 * SG, 3, rate, (double)sysID, (double)qsum(numAct), 0.0);
    }
    // accumulate for the averages
    double* sn1 = M.stress_n1 + 9 * bd.q_off + qo;
    double* hn1 = M.hist_n1 + bd.hist_off + qo;
#pragma unroll
    for (int k = 0; k < 6; k += 4) {
      const double v = qpick(sub, stress[k], stress[k + 1],
                             k + 2 < 6 ? stress[(k + 2) % 6] : 0.0,
                             k + 3 < 6 ? stress[(k + 3) % 6] : 0.0);
      double* w = sn1 + (k + sub) * SG;
      if (k + sub < 6) *w = c == 0 ? v : *w + v;
    }
#pragma unroll
    for (int i = 0; i < NSL; ++i) {
      double* w = hn1 + (75 + NSL * sub + i) * SG;
      *w = c == 0 ? slip[i] : *w + slip[i];
    }
#pragma unroll
    for (int i = 0; i < NSL; ++i) h1[(30 + NSL * sub + i) * SG] = slip[i];
  }
  if (cut) {
    atomicOr(&M.flags[1], 1);
    return;
  }
  const double rn = (double)ncry;
  const double* hn = fresh(hist_n);
  const double* sn9 = fresh(stress_n);
  const double* rot = rot_b ? fresh(rot_b) : nullptr;
  double* sn1 = M.stress_n1 + 9 * bd.q_off + qo;
  double* hn1 = M.hist_n1 + bd.hist_off + qo;
  double* cp = M.cep + 21 * bd.q_off + qo;
  t_work = t_work / rn;
  p_work = p_work / rn;
  p_strain = p_strain / rn;
  // mm10_a_store_crystal
#pragma unroll
  for (int k = 0; k < 6; k += 4)
    if (k + sub < 6) sn1[(k + sub) * SG] = sn1[(k + sub) * SG] / rn;
  // the tangent's average and [D] for the tangent kernel: the lower
  // triangle of history words 1-36
#pragma unroll
  for (int i = 0; i < 9; ++i) {
    const int k = sub + 4 * i, r = k % 6, cc = k / 6;
    const double v = hn1[k * SG] / rn;
    hn1[k * SG] = v;
    if (cc <= r) cp[(r * (r + 1) / 2 + cc) * SG] = v;
  }
#pragma unroll
  for (int i = 0; i < 7; ++i)
    if (sub + 4 * i < 27) hn1[(36 + sub + 4 * i) * SG] = 0.0;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const int k = sub + 4 * i;
    if (k < 9)
      hn1[(63 + k) * SG] = rot ? rot[k * SG] : ((k % 4 == 0) ? 1.0 : 0.0);
  }
  if (sub < 3) {  // energy, plastic work and strain
    const double v = qpick(sub, t_work, p_work, p_strain, 0.0);
    sn1[(6 + sub) * SG] = sn9[(6 + sub) * SG] + v;
    const double base = step == 1 ? 0.0 : hn[(72 + sub) * SG];
    hn1[(72 + sub) * SG] = base + v;
  }
#pragma unroll
  for (int i = 0; i < NSL; ++i) {
    const int64_t w = (75 + NSL * sub + i) * SG;
    double base = step == 1 ? 0.0 : hn[w];
    hn1[w] = base + hn1[w] / rn;
  }
}

// ---------------------------------------------------------------------
// grad Fe of mm10 blocks: rknstr_finish_cp (rknstr.f) with
// mm10_calc_grads (mm10_a.f:1579).  Small strains: for single-crystal
// elements the
// reference fits each component of Rt3d(3,3,ngp) linearly over the Gauss
// points (DGELS) and stores the three slopes of every component, the same
// 27 words at every point; Rt3d is a flat copy (mm10_a_copy_vector) of
// 9 ngp consecutive words of the block's gathered n-history
// elem_hist(span, hist, ngp) from (element 1, first Rp word of crystal 1,
// point 1), so words of several elements of the block enter it.  At step
// 1 those words are the values mm10 initialised in place.  Elements with
// several crystals get zeros.  Finite strains: per element (below).
// kGradWgs 256-lane workgroups per mm10 block, each fitting the block's 27
// words and writing its share of the points (a point per lane, so a word's
// stores are contiguous over the lanes).  Bound by the latency of the
// gather and fit, then by the 216 bytes a point: one 64-lane workgroup a
// block, which wrote the 27,648 words of 128 bricks alone, took 58 us.
// ---------------------------------------------------------------------
constexpr int kGradWgs = 8;
constexpr int kGradBlock = 256;
__device__ double mm10_init_word(const DevModel& M, const BlockDesc& bd,
                                 int w, int i, int64_t q, int64_t SG) {
  const double* hn = M.hist_n + bd.hist_off;
  if (w < kMM10Common)  // mm10_init_general_hist, _uout_hist, _slip_hist
    return (w >= 63 && w < 72) ? ((w - 63) % 4 == 0 ? 1.0 : 0.0) : 0.0;
  const int c = (w - kMM10Common) / kMM10Crystal;
  const int k = (w - kMM10Common) % kMM10Crystal;
  if (k < 6) return M.stress_n[9 * bd.q_off + k * SG + q];  // stress
  if (k < 9)                                                // angles
    return M.crys[bd.crys_off + (int64_t)i * bd.ncry + c].angles[k - 6];
  if (k < 18) return (k - 9) % 4 == 0 ? 1.0 : 0.0;          // Rp
  if (k == 42) return M.mats[bd.mat].cp.tau_y + 1.0e-5;     // tau tilde
  if (k < 58) return 0.0;
  return hn[w * SG + q];  // words mm10 does not initialise
}

__global__ void __launch_bounds__(kGradBlock)
    k_mm10_grads(DevModel M, const int32_t* __restrict__ blks, int lo,
                 int hi, int step) {
  const int b = blks[blockIdx.x / kGradWgs];
  if (b < lo || b >= hi) return;
  const BlockDesc bd = M.blocks[b];
  const GaussTable* gt = M.tables + bd.table;
  const int S = bd.span, G = bd.ngp, H = bd.hist;
  const int64_t SG = (int64_t)S * G;
  const int l = threadIdx.x;
  // the first point (or, for finite strains, element) of this lane
  const int first = (blockIdx.x % kGradWgs) * kGradBlock + l;
  if (first - l >= (bd.geonl ? S : (int)SG)) return;  // uniform
  __shared__ double s_v[9 * kMaxGp];
  __shared__ double s_g[27];
  const double* hn = M.hist_n + bd.hist_off;
  if (bd.ncry == 1) {
    for (int f = l; f < 9 * G; f += kGradBlock) {
      const int64_t L = (int64_t)(kMM10Common + 9) * S + f;
      const int i = (int)(L % S);
      const int w = (int)((L / S) % H);
      const int g = (int)(L / ((int64_t)S * H));
      const int64_t q = (int64_t)i * G + g;
      s_v[f] = step == 1 ? mm10_init_word(M, bd, w, i, q, SG) : hn[w * SG + q];
    }
  }
  __syncthreads();
  if (l < 27) {
    // grads(a, b, d) at a + 3b + 9d from Rt3d(a, b, p) at a + 3b + 9p
    double x = 0.0;
    if (bd.ncry == 1) {
      const int ab = l % 9, d = l / 9;
      for (int p = 0; p < G; ++p) x = x + gt->lsq[d][p] * s_v[ab + 9 * p];
    }
    s_g[l] = x;
  }
  __syncthreads();
  double* hn1 = M.hist_n1 + bd.hist_off;
  if (!bd.geonl) {
    for (int q = first; q < (int)SG; q += kGradWgs * kGradBlock)
#pragma unroll
      for (int k = 0; k < 27; ++k) hn1[(36 + k) * SG + q] = s_g[k];
    return;
  }
  // finite strains (mm10_calc_grads' geonl branch): per element, the fit
  // of Rp R^T (Rp of crystal 1 from the element's own n-history, R = [R
  // n+1]) taken to the current axes by the inverse (mm10_a_invert_33) of
  // the element's n = 0 Jacobian at its last point; zeros for several
  // crystals or a singular Jacobian
  for (int i = first; i < S; i += kGradWgs * kGradBlock) {
    double gv[27];
#pragma unroll
    for (int k = 0; k < 27; ++k) gv[k] = 0.0;
    const double* a = M.jac_tmp + 9 * ((int64_t)bd.felem - 1 + i);
#define A3(r, c) a[3 * ((r)-1) + (c)-1]
    const double det =
        A3(1, 1) * A3(2, 2) * A3(3, 3) - A3(1, 1) * A3(2, 3) * A3(3, 2) -
        A3(1, 2) * A3(2, 1) * A3(3, 3) + A3(1, 2) * A3(2, 3) * A3(3, 1) +
        A3(1, 3) * A3(2, 1) * A3(3, 2) - A3(1, 3) * A3(2, 2) * A3(3, 1);
    if (bd.ncry == 1 && fabs(det) > 1.0e-10) {
      double ji[9];  // jacinv row-major: transpose(cofactor) / det
      ji[0] = (A3(2, 2) * A3(3, 3) - A3(2, 3) * A3(3, 2)) / det;
      ji[3] = -(A3(2, 1) * A3(3, 3) - A3(2, 3) * A3(3, 1)) / det;
      ji[6] = (A3(2, 1) * A3(3, 2) - A3(2, 2) * A3(3, 1)) / det;
      ji[1] = -(A3(1, 2) * A3(3, 3) - A3(1, 3) * A3(3, 2)) / det;
      ji[4] = (A3(1, 1) * A3(3, 3) - A3(1, 3) * A3(3, 1)) / det;
      ji[7] = -(A3(1, 1) * A3(3, 2) - A3(1, 2) * A3(3, 1)) / det;
      ji[2] = (A3(1, 2) * A3(2, 3) - A3(1, 3) * A3(2, 2)) / det;
      ji[5] = -(A3(1, 1) * A3(2, 3) - A3(1, 3) * A3(2, 1)) / det;
      ji[8] = (A3(1, 1) * A3(2, 2) - A3(1, 2) * A3(2, 1)) / det;
#undef A3
      double sl[27];  // slopes (d) of component (a, b) at a + 3 b + 9 d
#pragma unroll
      for (int k = 0; k < 27; ++k) sl[k] = 0.0;
      for (int g = 0; g < G; ++g) {
        const int64_t q = (int64_t)i * G + g;
        double Rp[9], R[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) {
          const int w = kMM10Common + 9 + k;  // Rp of crystal 1
          Rp[k] = step == 1 ? mm10_init_word(M, bd, w, i, q, SG)
                            : hn[w * SG + q];
          R[k] = M.rot_tmp[9 * bd.q_off + k * SG + q];
        }
#pragma unroll
        for (int ia = 0; ia < 3; ++ia)
#pragma unroll
          for (int ib = 0; ib < 3; ++ib) {
            // mm10_a_mult_type_3t: (Rp R^T)(ia, ib)
            const double v = Rp[ia] * R[ib] + Rp[ia + 3] * R[ib + 3] +
                             Rp[ia + 6] * R[ib + 6];
#pragma unroll
            for (int d = 0; d < 3; ++d)
              sl[ia + 3 * ib + 9 * d] = sl[ia + 3 * ib + 9 * d] +
                                        gt->lsq[d][g] * v;
          }
      }
#pragma unroll
      for (int ab = 0; ab < 9; ++ab)
#pragma unroll
        for (int d = 0; d < 3; ++d)
          gv[ab + 9 * d] = ji[3 * d] * sl[ab] + ji[3 * d + 1] * sl[ab + 9] +
                           ji[3 * d + 2] * sl[ab + 18];
    }
    for (int g = 0; g < G; ++g) {
      const int64_t q = (int64_t)i * G + g;
#pragma unroll
      for (int k = 0; k < 27; ++k) hn1[(36 + k) * SG + q] = gv[k];
    }
  }
}

int launch_mm10_grads(const DevModel& M, const int32_t* d_blks, int nblks,
                      int lo, int hi, int step, hipStream_t s) {
  if (nblks > 0)
    hipLaunchKernelGGL(k_mm10_grads, dim3(nblks * kGradWgs), dim3(kGradBlock),
                       0, s, M, d_blks, lo, hi, step);
  return hipGetLastError() == hipSuccess ? W3D_OK : W3D_ERR_DEVICE;
}

// Persistent over the work list: each workgroup (one wave) takes the next
// part of kPts points of a work item from a device counter until the list
// is exhausted, so points whose local solves sub-step or iterate longer do
// not hold back a fixed share of the grid.  The counter starts at zero
// (launch_mm10 clears it with a fill kernel first).
constexpr int kItemParts = 64 / kPts;  // parts of a 64-point item

__global__ void __launch_bounds__(64)
    __attribute__((amdgpu_waves_per_eu(2)))
    k_mm10(DevModel M, const WorkItem* __restrict__ work, int nwork,
           int* __restrict__ counter, int step, int iter0_off) {
  __shared__ double s_mem[kMemWords];
  __shared__ int s_item;
  for (;;) {
    if (threadIdx.x == 0) s_item = atomicAdd(counter, 1);
    __syncthreads();
    const int unit = __builtin_amdgcn_readfirstlane(s_item);
    __syncthreads();
    if (unit >= kItemParts * nwork) break;  // uniform across the workgroup
    mm10_item(M, work[unit / kItemParts], unit % kItemParts, step, iter0_off,
              s_mem);
  }
}

// The batched form: the items of every slot in one list, slot s owning
// global items [item0_s, item0_s + nwork_s); the workgroup finds its slot
// by bisection over the slots' item0 (ascending).
__global__ void __launch_bounds__(64)
    __attribute__((amdgpu_waves_per_eu(2)))
    k_mm10_batch(const Mm10Slot* __restrict__ slots, int nslot,
                 int nwork_total, int* __restrict__ counter) {
  __shared__ double s_mem[kMemWords];
  __shared__ int s_item;
  for (;;) {
    if (threadIdx.x == 0) s_item = atomicAdd(counter, 1);
    __syncthreads();
    const int unit = __builtin_amdgcn_readfirstlane(s_item);
    __syncthreads();
    if (unit >= kItemParts * nwork_total) break;  // uniform
    const int item = unit / kItemParts;
    int lo = 0, hi = nslot - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (slots[mid].item0 <= item)
        lo = mid;
      else
        hi = mid - 1;
    }
    const Mm10Slot& sl = slots[lo];
    mm10_item(sl.M, sl.work[item - sl.item0], unit % kItemParts, sl.step,
              sl.iter0_off, s_mem);
  }
}

int launch_mm10_batch(const Mm10Slot* d_slots, int nslot, int nwork_total,
                      int* d_counter, int grid, hipStream_t s) {
  if (nwork_total <= 0 || nslot <= 0) return W3D_OK;
  int rc = launch_fill_i32(d_counter, 1, 0, s);
  if (rc) return rc;
  hipLaunchKernelGGL(k_mm10_batch,
                     dim3(std::min(grid, kItemParts * nwork_total)), dim3(64),
                     0, s, d_slots, nslot, nwork_total, d_counter);
  return hipGetLastError() == hipSuccess ? W3D_OK : W3D_ERR_DEVICE;
}

int launch_mm10(const DevModel& M, const WorkItem* d_work, int nwork,
                int* d_counter, int grid, int step, int iter0_off,
                hipStream_t s) {
  if (nwork <= 0) return W3D_OK;
  int rc = launch_fill_i32(d_counter, 1, 0, s);
  if (rc) return rc;
  hipLaunchKernelGGL(k_mm10, dim3(std::min(grid, kItemParts * nwork)),
                     dim3(64), 0, s, M, d_work, nwork, d_counter, step,
                     iter0_off);
  return hipGetLastError() == hipSuccess ? W3D_OK : W3D_ERR_DEVICE;
}

}  // namespace w3d
