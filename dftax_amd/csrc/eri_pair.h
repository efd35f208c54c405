// Device pieces shared by the bra-pair kernels (eri_pair.hip: integrals, eri_pair_grad.hip: their
// nuclear derivatives): the one-axis Hermite tables, the R ladder by planes, the bra description.
#pragma once

#include <cstdint>

#include "dfks_common.h"

namespace dfks {

namespace {

typedef double dbl4 __attribute__((ext_vector_type(4)));

__host__ __device__ constexpr int n_tet(int L) { return (L + 1) * (L + 2) * (L + 3) / 6; }

// cart->sph lists and cartesian exponents, a copy per translation unit (filled by its upload function)
__constant__ C2SList g_c2s_pair;
__constant__ int g_cart_pair[7][28][3];

// E^{ij}_t of one axis into E[(i (LB+1) + j) (LAB+1) + t], zero where t > i + j
template <int LA, int LB>
__device__ __forceinline__ void e_axis(double xpa, double xpb, double i2p, double* __restrict__ out) {
  constexpr int MT = LA + LB + 1;
  double E[LA + 1][LB + 1][MT];
#pragma unroll
  for (int i = 0; i <= LA; ++i)
#pragma unroll
    for (int j = 0; j <= LB; ++j)
#pragma unroll
      for (int t = 0; t < MT; ++t) E[i][j][t] = 0.0;
  E[0][0][0] = 1.0;
#pragma unroll
  for (int i = 0; i < LA; ++i)
#pragma unroll
    for (int t = 0; t <= i + 1; ++t) {
      double v = xpa * E[i][0][t];
      if (t > 0) v += i2p * E[i][0][t - 1];
      if (t + 1 <= i) v += (t + 1) * E[i][0][t + 1];
      E[i + 1][0][t] = v;
    }
#pragma unroll
  for (int j = 0; j < LB; ++j)
#pragma unroll
    for (int i = 0; i <= LA; ++i)
#pragma unroll
      for (int t = 0; t <= i + j + 1; ++t) {
        double v = xpb * E[i][j][t];
        if (t > 0) v += i2p * E[i][j][t - 1];
        if (t + 1 <= i + j) v += (t + 1) * E[i][j][t + 1];
        E[i][j + 1][t] = v;
      }
#pragma unroll
  for (int i = 0; i <= LA; ++i)
#pragma unroll
    for (int j = 0; j <= LB; ++j)
#pragma unroll
      for (int t = 0; t < MT; ++t) out[(i * (LB + 1) + j) * MT + t] = E[i][j][t];
}

// One plane v of R: the (t,u) triangle of order <= TOP by the in-place ladder from Z[n] = R^(n)_00v
template <int TOP>
__device__ __forceinline__ void r_plane(double x, double y, const double* Z, double* X) {
  X[0] = Z[TOP];
#pragma unroll
  for (int m = TOP - 1; m >= 0; --m) {
#pragma unroll
    for (int r = TOP - m; r >= 1; --r)
#pragma unroll
      for (int u = 0; u <= r; ++u) {
        const int t = r - u, e = r * (r + 1) / 2 + u;
        if (t > 0) {
          double v = x * X[(r - 1) * r / 2 + u];
          if (t > 1) v += (t - 1) * X[(r - 2) * (r - 1) / 2 + u];
          X[e] = v;
        } else {
          double v = y * X[(r - 1) * r / 2 + u - 1];
          if (u > 1) v += (u - 1) * X[(r - 2) * (r - 1) / 2 + u - 2];
          X[e] = v;
        }
      }
    X[0] = Z[m];
  }
}

// Planes v = V0 + sub of this lane, then V0 + 4 + sub, ...: ladder in registers, entries of order
// LC .. L to Rw[index - R0][16 lanes]
template <int L, int LC, int R0, int V0>
__device__ __forceinline__ void r_planes(double x, double y, double z, int v, double* Zc, double* Zp,
                                         double* __restrict__ Rw) {
  if constexpr (V0 <= L) {
    constexpr int TOP = L - V0;
    double X[(TOP + 1) * (TOP + 2) / 2];
    r_plane<TOP>(x, y, Zc, X);
    const int vb = v * (v + 1) / 2 + v - R0;
#pragma unroll
    for (int r = 0; r <= TOP; ++r) {
      const int s = r + v;
      if (s >= LC && s <= L) {
        double* dst = Rw + (s * (s + 1) * (s + 2) / 6 + vb) * 16;
#pragma unroll
        for (int u = 0; u <= r; ++u) dst[(u * (u + 1) / 2 + u * v) * 16] = X[r * (r + 1) / 2 + u];
      }
    }
    if constexpr (V0 + 4 <= L) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const double fv = (double)(v + k);
#pragma unroll
        for (int n = 0; n + V0 < L; ++n) {
          const double nz = z * Zc[n + 1] + fv * Zp[n + 1];
          Zp[n] = Zc[n];
          Zc[n] = nz;
        }
      }
      r_planes<L, LC, R0, V0 + 4>(x, y, z, v + 4, Zc, Zp, Rw);
    }
  }
}

// The bra shell pair: its primitives' slices and centres. A single shell (the bra of the two-centre
// integrals) has the unit function of exponent 0 at its own centre for a partner.
struct BraPair {
  const double *ea, *eb, *ca, *cb;
  const double *xa, *xb;
  int npb;
};
__constant__ double g_unit_exp[1] = {0.0}, g_unit_coef[1] = {1.0};

__device__ __forceinline__ BraPair bra_pair(const ShellSet& A, int ia, int ib, bool unit) {
  const double *ea = A.exps + A.prim0[ia], *ca = A.coefs + A.prim0[ia], *xa = A.centre + 3 * ia;
  if (unit) return {ea, g_unit_exp, ca, g_unit_coef, xa, xa, 1};
  return {ea, A.exps + A.prim0[ib], ca, A.coefs + A.prim0[ib], xa, A.centre + 3 * ib, A.nprim[ib]};
}

}  // namespace

}  // namespace dfks
