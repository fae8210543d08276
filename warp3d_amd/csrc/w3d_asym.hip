// w3d_asym.hip -- asymmetric assembly: the full element matrices and their
// gather into full CSR rows, FP64.
//
// Reference: gptns1.f:1513 bdbt_asym (BD(j,k) = sum_m D(m,k) B(m,j), then
// ek_full(j) += sum_r B(r,col) BD(row,r) for j = (col-1) T + row, every
// row and column), gptns1.f:1371 drive_10_cnst ([D] = the point's history
// words 1-36, column-major, times w |J|), gptns1.f:1174 extract_D_symmetric
// (mm01), gpmas1.f:399 adjust_cnst (1/6 for tets), assemble_code.f:1050
// assem_by_row_asymmetric / assem_a_row_asym (row srow gathers the words
// (erow-1) T + ecol of each element on its node, elements in
// inverse-incidence order, the column found by binary search).
//
// The full matrices themselves are formed on the matrix cores
// (w3d_tangent.hip).  The assembly runs one wave per row group (the free
// equations of one node) over a map built once per pattern: for each (node,
// element) incidence, the Ke base of the element and, per element column,
// its position in the CSR rows of the node (the same for the node's three
// rows), or none if constrained.
#include <hip/hip_runtime.h>

#include "w3d_internal.h"
#include "w3d_wave.h"

namespace w3d {

// One wave per row group: the node's rows (at most 3, one after the other
// in the CSR and of one length) are summed in LDS, element after element in
// inverse-incidence order, a lane adding the element's word (erow-1) T +
// ecol of one (row, ecol) pair (distinct columns within an element, so no
// two lanes meet); an element row's Ke words and the group's values are read
// and written contiguously.
// Bound by the chain of dependent loads of a wave (group, node, incidences,
// positions and Ke words).  A wave per equation row walked it three times a
// node, with 24 of the 64 lanes at work on bricks, and its fixed 768-word
// row held a CU to 24 waves; the rows' LDS is now the pattern's longest row
// (21,924 bricks: 110 -> 62 us, 2.3 TB/s of Ke words and values).
constexpr int kAsmWaves = 4;
constexpr int kAsmChunk = 4;  // elements whose loads are in flight together
constexpr int kAsmRounds = (3 * kMaxDof + 63) / 64;  // (row, ecol) pairs

__global__ void __launch_bounds__(64 * kAsmWaves)
    k_assemble_full(const double* __restrict__ ekf,
                    const int64_t* __restrict__ ebase,
                    const int64_t* __restrict__ atoff,
                    const uint16_t* __restrict__ at,
                    const int32_t* __restrict__ eq_dof,
                    const int64_t* __restrict__ inv_ptr,
                    const int32_t* __restrict__ inv_ln, RowGroups A,
                    int maxrow, double* __restrict__ val) {
  extern __shared__ double s_rows[];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int g = blockIdx.x * (blockDim.x >> 6) + wv;
  if (g >= A.ngrp) return;  // uniform across the wave
  const RowGroup gd = A.grp[g];
  const int r0 = gd.row0, nr = gd.rows();
  const int64_t v0 = gd.k0;
  const int len = gd.len();  // <= maxrow
  double* row = s_rows + (size_t)wv * 3 * maxrow;
  for (int k = lane; k < nr * len; k += 64) row[k] = 0.0;
  wave_sync();
  const int d0 = eq_dof[r0], node = d0 / 3;
  const int comp0 = d0 % 3;
  const int comp1 = nr > 1 ? eq_dof[r0 + 1] % 3 : 0;
  const int comp2 = nr > 2 ? eq_dof[r0 + 2] % 3 : 0;
  const int64_t pb = inv_ptr[node], pe = inv_ptr[node + 1];
  // elements in chunks of kAsmChunk: their loads are independent and
  // overlap; the sums then go into LDS in element order
  for (int64_t p0 = pb; p0 < pe; p0 += kAsmChunk) {
    int pos[kAsmChunk][kAsmRounds];
    double v[kAsmChunk][kAsmRounds];
#pragma unroll
    for (int j = 0; j < kAsmChunk; ++j) {
      const int64_t p = p0 + j;
#pragma unroll
      for (int m = 0; m < kAsmRounds; ++m) {
        pos[j][m] = -1;
        v[j][m] = 0.0;
      }
      if (p >= pe) continue;
      const int64_t a0 = atoff[p];
      const int T = (int)(atoff[p + 1] - a0);
      const int ln = inv_ln[p];
      const double* ke = ekf + ebase[p];
#pragma unroll
      for (int m = 0; m < kAsmRounds; ++m) {
        if (64 * m >= nr * T) continue;  // uniform
        const int x = lane + 64 * m;
        if (x >= nr * T) continue;
        const int k = (x >= T ? 1 : 0) + (x >= 2 * T ? 1 : 0);
        const int ecol = x - k * T;
        const int at_p = at[a0 + ecol];
        if (at_p == kAsmNone) continue;
        const int comp = k == 0 ? comp0 : k == 1 ? comp1 : comp2;
        pos[j][m] = k * len + at_p;
        v[j][m] = ke[(comp * (T / 3) + ln) * T + ecol];
      }
    }
#pragma unroll
    for (int j = 0; j < kAsmChunk; ++j) {
#pragma unroll
      for (int m = 0; m < kAsmRounds; ++m)
        if (pos[j][m] >= 0) row[pos[j][m]] = row[pos[j][m]] + v[j][m];
      wave_sync();
    }
  }
  for (int k = lane; k < nr * len; k += 64) val[v0 + k] = row[k];
}

int launch_assemble_full(const double* ekf, const int64_t* ebase,
                         const int64_t* atoff, const uint16_t* at,
                         const int32_t* eq_dof, const int64_t* inv_ptr,
                         const int32_t* inv_ln, const RowGroups& A,
                         int maxrow, double* val, hipStream_t s) {
  if (A.ngrp == 0) return W3D_OK;
  // four waves a workgroup while their rows fit 64 KB of LDS (rows of up
  // to 682 entries), else two (kAsmMaxRow: 37 KB)
  const int waves = kAsmWaves * 3 * maxrow * 8 <= 65536 ? kAsmWaves : 2;
  hipLaunchKernelGGL(k_assemble_full, dim3((A.ngrp + waves - 1) / waves),
                     dim3(64 * waves), (size_t)waves * 3 * maxrow * 8, s, ekf,
                     ebase, atoff, at, eq_dof, inv_ptr, inv_ln, A, maxrow,
                     val);
  return hipGetLastError() == hipSuccess ? W3D_OK : W3D_ERR_DEVICE;
}

}  // namespace w3d
