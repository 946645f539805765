// rism_chi.h -- chi_vv(|k|) tables of the OZ step, shared by the x pass and the
// plane pass.
#pragma once
#include "rism_common.h"

namespace rism {

// chi_vv(|k|) sources for the OZ step.  ChiTable: a table built once per context, one row of natv^2 values per k^2 shell for a cubic box
// (k_chi_table), or one per point of the octant kx, ky, kz > 0 for a box with
// different sides (k_chi_octant; |k| has few repeats there).
// The octant table holds natv^2 / 8 words per grid point, which the pass
// reads once a step, and against it stood four coefficient gathers, a square
// root and a knot search per k and pair of sites: 144 x 160 x 128, 4 sites,
// 124 -> 79 us; 72 x 90 x 60, 2 sites, 17 -> 9 us.
template <class Tb, int STRIDE>
struct ChiTable {
  const Tb *row;
  __device__ __forceinline__ Tb operator()(int pw) const { return row[pw * STRIDE]; }
};
// the table's row for the points (+-kx, +-ky) at x index jx < L/2, y index
// yh < ny/2 and plane m.  Shells are rows of consecutive values; in the
// octant the x index is fastest, so that neighbouring threads read
// neighbouring words.
template <int L, int CHI, class Tb>
__device__ __forceinline__ auto chi_row(const Tb *tab, const Params &P, int nv2, int jx, int yh,
                                        int m) {
  if constexpr (CHI == RISM_CHI_OCTANT) {
    return ChiTable<Tb, L / 2>{tab + ((size_t)m * (P.ny / 2) + yh) * nv2 * (L / 2) + jx};
  } else {
    // |k|^2 = (pi/L)^2 (8 sidx + 3)
    const long ox = 2 * jx - L + 1, oy = 2 * yh - P.ny + 1, oz = 2 * m + 1;
    const long sidx = (ox * ox + oy * oy + oz * oz - 3) >> 3;
    return ChiTable<Tb, 1>{tab + sidx * nv2};
  }
}

// OZ at two points that share |k|, (kx, ky) and (-kx, ky) of one row, with
// their chi row in registers (chr[v][w], v, w < NV): H_v = sum_w X[v][w] (C_w -
// q_w fk) (mqvfk + oz, calculate_cuda.cu:32-52).  off[k] is the LDS offset of
// point k in site 0's values; site w sits w*CS further.
template <int NV, int NVM, class Re>
__device__ __forceinline__ void oz_points_reg(cx<Re> *lds, int CS, const int (&off)[2],
                                              const cx<Re> (&fk)[2], const Params &P,
                                              const Re (&chr)[NVM][NVM]) {
  cx<Re> c[2][NV];
#pragma unroll
  for (int w = 0; w < NV; ++w) {
#pragma unroll
    for (int k = 0; k < 2; ++k) c[k][w] = lds[off[k] + w * CS] - (Re)P.qv[w] * fk[k];
  }
#pragma unroll
  for (int v = 0; v < NV; ++v) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      cx<Re> a{0, 0};
#pragma unroll
      for (int w = 0; w < NV; ++w) a = a + chr[v][w] * c[k][w];
      lds[off[k] + v * CS] = a;
    }
  }
}

}  // namespace rism
