// One-electron integrals and their nuclear derivatives by shell pair: one wavefront per pair, one
// template instance per class (l_a >= l_b), any span.
//
// Nuclear attraction is sum_h H[ab][h] S[h] with S[h] = sum_C -Z_C 2 pi / p R_h(P - C): the nuclei are
// summed before the pair's Hermite coefficients are met, 16 of them at a time, 4 lanes each (R by
// planes as in eri_pair.hip). Its derivative weights are N[h] = sum_ab P_ab H[ab][h] and the same
// with dH/dX, X = A - B, so that per nucleus only the sums of N R_{h+x} and of dN R_h are formed
// (d/dA = (a/p) d/dP + d/dX, d/dB = (b/p) d/dP - d/dX, d/dC = -d/dP). S and T come from the one-axis
// tables. What bounds it is the chain of one primitive pair: tables, nuclei, contraction.
// Against a wavefront per ordered pair that met one nucleus at a time, lane 0 on the Boys function:
// S, T and V of (H2O)_8 def2-TZVP 0.46 ms (2.6); the gradient of a 6-heavy-atom tree, def2-SVP, with
// its four energy-weighted densities in one pass 1.0 ms (15 in four).
// Reference: dftax/integrals (overlap, kinetic, nuclear), dftax/ks/forces.py:128-270.
#include <cstdint>

#include "eri_pair.h"

namespace dfks {

namespace {

// h -> (t, u, v) packed 4 bits each
__device__ __forceinline__ int pack_tuv(int h) {
  int s = 0;
  while (h >= n_tet(s)) ++s;
  const int k = h - (s > 0 ? n_tet(s - 1) : 0);
  int r = 0;
  while (k >= (r + 1) * (r + 2) / 2) ++r;
  const int v = k - r * (r + 1) / 2;
  return (s - r) | ((r - v) << 4) | (v << 8);
}

// R_h(P - C) of order <= L of 16 nuclei (lane % 16, from c0) into R[h][16], weighted by -Z f; lanes past the
// last nucleus weigh 0
template <int L>
__device__ __forceinline__ void nuclear_r(int c0, int natm, const double* __restrict__ atm, double f, double p,
                                          double Px, double Py, double Pz, const double* __restrict__ boys,
                                          double* __restrict__ R) {
  const int lane = threadIdx.x & 63, ax = lane & 15, sub = lane >> 4;
  const int c = min(c0 + ax, natm - 1);
  double pref = c0 + ax < natm ? -atm[4 * c + 3] * f : 0.0;
  const double x = Px - atm[4 * c], y = Py - atm[4 * c + 1], z = Pz - atm[4 * c + 2];
  double Zc[L + 1], Zp[L + 1];
  boys_array<L>(p * (x * x + y * y + z * z), Zc, boys);
  const double n2r = -2.0 * p;
#pragma unroll
  for (int n = 0; n <= L; ++n) {
    Zc[n] *= pref;
    pref *= n2r;
    Zp[n] = 0.0;
  }
#pragma unroll
  for (int k = 0; k < 3 && k < L; ++k) {
    const bool go = k < sub;
#pragma unroll
    for (int n = 0; n + k < L; ++n) {
      const double nz = z * Zc[n + 1] + (double)k * Zp[n + 1];
      Zp[n] = go ? Zc[n] : Zp[n];
      Zc[n] = go ? nz : Zc[n];
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  r_planes<L, 0, 0, 0>(x, y, z, sub, Zc, Zp, R + ax);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

template <int LA, int LB>
__global__ __launch_bounds__(64) void k_int1e(const int2* __restrict__ pairs, ShellSet A, int natm,
                                              const double* __restrict__ atm, const double* __restrict__ boys,
                                              double* __restrict__ S, double* __restrict__ Tm, double* __restrict__ V,
                                              int64_t nao) {
  constexpr int LAB = LA + LB, NA = ncart(LA), NB = ncart(LB), NO = NA * NB, EJ = LB + 3, MT = LAB + 3;
  constexpr int NH = n_tet(LAB), HQ = (NH + 3) / 4;
  __shared__ double s_E[3][(LA + 1) * EJ * MT];
  __shared__ double s_c[3][NO];
  __shared__ double s_R[NH * 16];
  __shared__ double s_S[NH];
  const int lane = threadIdx.x, ax = lane & 15, sub = lane >> 4;
  const int2 pr = pairs[blockIdx.x];
  const int ia = pr.x, ib = pr.y;
  const double *xa = A.centre + 3 * ia, *xb = A.centre + 3 * ib;
  const double dx = xa[0] - xb[0], dy = xa[1] - xb[1], dz = xa[2] - xb[2], ab2 = dx * dx + dy * dy + dz * dz;
  for (int o = lane; o < 3 * NO; o += 64) (&s_c[0][0])[o] = 0.0;
  for (int pa = 0; pa < A.nprim[ia]; ++pa)
    for (int pb = 0; pb < A.nprim[ib]; ++pb) {
      const double al = A.exps[A.prim0[ia] + pa], be = A.exps[A.prim0[ib] + pb];
      const double p = al + be, ip = 1.0 / p;
      const double cab = A.coefs[A.prim0[ia] + pa] * A.coefs[A.prim0[ib] + pb] * exp(-al * be * ip * ab2);
      __syncthreads();
      if (lane < 3) {
        const double ab = xa[lane] - xb[lane];
        e_axis<LA, LB + 2>(-be * ab * ip, al * ab * ip, 0.5 * ip, s_E[lane]);
      }
      __syncthreads();
      const double s0 = kPi * ip * sqrt(kPi * ip) * cab;
      for (int o = lane; o < NO; o += 64) {
        const int ai = o / NB, bi = o % NB;
        double s1[3], t1[3];
#pragma unroll
        for (int x = 0; x < 3; ++x) {
          const int i = g_cart_pair[LA][ai][x], j = g_cart_pair[LB][bi][x];
          const double* E = s_E[x] + i * EJ * MT;
          const double sij = E[j * MT];
          double tt = -2.0 * be * be * E[(j + 2) * MT] + be * (2 * j + 1) * sij;
          if (j >= 2) tt -= 0.5 * j * (j - 1) * E[(j - 2) * MT];
          s1[x] = sij;
          t1[x] = tt;
        }
        s_c[0][o] += s0 * s1[0] * s1[1] * s1[2];
        s_c[1][o] += s0 * (t1[0] * s1[1] * s1[2] + s1[0] * t1[1] * s1[2] + s1[0] * s1[1] * t1[2]);
      }
      if (natm == 0) continue;
      double acc[HQ];
#pragma unroll
      for (int q = 0; q < HQ; ++q) acc[q] = 0.0;
      const double Px = (al * xa[0] + be * xb[0]) * ip, Py = (al * xa[1] + be * xb[1]) * ip,
                   Pz = (al * xa[2] + be * xb[2]) * ip;
      for (int c0 = 0; c0 < natm; c0 += 16) {
        nuclear_r<LAB>(c0, natm, atm, cab * 2.0 * kPi * ip, p, Px, Py, Pz, boys, s_R);
#pragma unroll
        for (int q = 0; q < HQ; ++q) acc[q] += s_R[min(4 * q + sub, NH - 1) * 16 + ax];
      }
#pragma unroll
      for (int q = 0; q < HQ; ++q) {
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) acc[q] += __shfl_xor(acc[q], o, 16);
        if (ax == 0 && 4 * q + sub < NH) s_S[4 * q + sub] = acc[q];
      }
      __syncthreads();
      for (int o = lane; o < NO; o += 64) {
        const int ai = o / NB, bi = o % NB;
        int m[3];
        const double* E[3];
#pragma unroll
        for (int x = 0; x < 3; ++x) {
          const int i = g_cart_pair[LA][ai][x], j = g_cart_pair[LB][bi][x];
          m[x] = i + j;
          E[x] = s_E[x] + (i * EJ + j) * MT;
        }
        double sum = 0.0;
        for (int t = 0; t <= m[0]; ++t)
          for (int u = 0; u <= m[1]; ++u) {
            const double e = E[0][t] * E[1][u];
            for (int v = 0; v <= m[2]; ++v) {
              const int s = t + u + v, r = u + v;
              sum += e * E[2][v] * s_S[s * (s + 1) * (s + 2) / 6 + r * (r + 1) / 2 + v];
            }
          }
        s_c[2][o] += sum;
      }
    }
  __syncthreads();
  const bool sphA = A.spherical && LA >= 2, sphB = A.spherical && LB >= 2;
  const int fa = sphA ? nsph(LA) : NA, fb = sphB ? nsph(LB) : NB;
  for (int o = lane; o < fa * fb; o += 64) {
    const int Ai = o / fb, Bi = o % fb;
    const int nA = sphA ? g_c2s_pair.n[LA][Ai] : 1, nB = sphB ? g_c2s_pair.n[LB][Bi] : 1;
    double v[3] = {0.0, 0.0, 0.0};
    for (int x = 0; x < nA; ++x) {
      const int ai = sphA ? g_c2s_pair.cart[LA][Ai][x] : Ai;
      const double wa = sphA ? g_c2s_pair.coef[LA][Ai][x] : 1.0;
      for (int y = 0; y < nB; ++y) {
        const int bi = sphB ? g_c2s_pair.cart[LB][Bi][y] : Bi;
        const double w = wa * (sphB ? g_c2s_pair.coef[LB][Bi][y] : 1.0);
#pragma unroll
        for (int z = 0; z < 3; ++z) v[z] += w * s_c[z][ai * NB + bi];
      }
    }
    const int64_t i1 = (int64_t)(A.ao0[ia] + Ai) * nao + A.ao0[ib] + Bi;
    const int64_t i2 = (int64_t)(A.ao0[ib] + Bi) * nao + A.ao0[ia] + Ai;
    S[i1] = S[i2] = v[0];
    Tm[i1] = Tm[i2] = v[1];
    V[i1] = V[i2] = v[2];
  }
}

// The block M[a, b] of a symmetric matrix to cartesian components, by one wavefront
template <int LA, int LB>
__device__ __forceinline__ void block_to_cart(const double* __restrict__ M, int64_t nao, int a0, int b0, int sph,
                                              double* __restrict__ out) {
  constexpr int NA = ncart(LA), NB = ncart(LB);
  const bool sphA = sph && LA >= 2, sphB = sph && LB >= 2;
  const int fa = sphA ? nsph(LA) : NA, fb = sphB ? nsph(LB) : NB;
  for (int o = threadIdx.x; o < NA * NB; o += 64) {
    double v = 0.0;
    const int ai = o / NB, bi = o % NB;
    for (int x = 0; x < fa; ++x) {
      double wa = x == ai ? 1.0 : 0.0;
      if (sphA) {
        wa = 0.0;
        for (int k = 0; k < g_c2s_pair.n[LA][x]; ++k)
          if (g_c2s_pair.cart[LA][x][k] == ai) wa = g_c2s_pair.coef[LA][x][k];
      }
      if (wa == 0.0) continue;
      for (int y = 0; y < fb; ++y) {
        double wb = y == bi ? 1.0 : 0.0;
        if (sphB) {
          wb = 0.0;
          for (int k = 0; k < g_c2s_pair.n[LB][y]; ++k)
            if (g_c2s_pair.cart[LB][y][k] == bi) wb = g_c2s_pair.coef[LB][y][k];
        }
        if (wb != 0.0) v += wa * wb * M[(int64_t)(a0 + x) * nao + b0 + y];
      }
    }
    out[o] = v;
  }
}

// grad[0] += sum P d(T + V) - W_0 dS, grad[k] -= W_k dS (k = 1..3), all [natm][3], natm3 = 3 natm words apart;
// unordered pairs, off-diagonal ones twice. W: 4 matrices, nao^2 apart by pointer.
struct Int1eW {
  const double* w[4];
};
template <int LA, int LB>
__global__ __launch_bounds__(64) void k_int1e_pgrad(const int2* __restrict__ pairs, ShellSet A,
                                                    const int32_t* __restrict__ atom_a, int natm,
                                                    const double* __restrict__ atm, const double* __restrict__ boys,
                                                    const double* __restrict__ P, Int1eW W, int64_t nao,
                                                    double* __restrict__ grad, int64_t part) {
  constexpr int LAB = LA + LB, L = LAB + 1, NA = ncart(LA), NB = ncart(LB), NO = NA * NB, EJ = LB + 3, MT = LAB + 4;
  constexpr int NH = n_tet(LAB), HQ = (NH + 3) / 4;
  __shared__ double s_E[3][(LA + 2) * EJ * MT];
  __shared__ double s_w[5][NO];          // P, W_0 .. W_3 in cartesian components
  __shared__ double s_N[4][NH];
  __shared__ int s_h[NH];
  __shared__ double s_R[n_tet(L) * 16];
  const int lane = threadIdx.x, ax = lane & 15, sub = lane >> 4;
  const int2 pr = pairs[blockIdx.x];
  const int ia = pr.x, ib = pr.y;
  const double *xa = A.centre + 3 * ia, *xb = A.centre + 3 * ib;
  const double dx = xa[0] - xb[0], dy = xa[1] - xb[1], dz = xa[2] - xb[2], ab2 = dx * dx + dy * dy + dz * dz;
  const double f = ia != ib ? 2.0 : 1.0;
  block_to_cart<LA, LB>(P, nao, A.ao0[ia], A.ao0[ib], A.spherical, s_w[0]);
#pragma unroll
  for (int k = 0; k < 4; ++k) block_to_cart<LA, LB>(W.w[k], nao, A.ao0[ia], A.ao0[ib], A.spherical, s_w[1 + k]);
  for (int h = lane; h < NH; h += 64) s_h[h] = pack_tuv(h);
  double gS[4][3] = {}, gA[3] = {}, gB[3] = {};
  for (int pa = 0; pa < A.nprim[ia]; ++pa)
    for (int pb = 0; pb < A.nprim[ib]; ++pb) {
      const double al = A.exps[A.prim0[ia] + pa], be = A.exps[A.prim0[ib] + pb];
      const double p = al + be, ip = 1.0 / p;
      const double cab = A.coefs[A.prim0[ia] + pa] * A.coefs[A.prim0[ib] + pb] * exp(-al * be * ip * ab2);
      __syncthreads();
      if (lane < 3) e_table_1d(LA + 1, LB + 2, al, be, xa[lane] - xb[lane], MT, s_E[lane]);
      __syncthreads();
      const double s0 = kPi * ip * sqrt(kPi * ip) * cab;
      // overlap and kinetic: the bra derivative 2a f_{i+1,j} - i f_{i-1,j}; the ket's is its negative
      for (int o = lane; o < NO; o += 64) {
        const int ai = o / NB, bi = o % NB;
        double s1[3], t1[3], ds[3], dt[3];
#pragma unroll
        for (int x = 0; x < 3; ++x) {
          const int i = g_cart_pair[LA][ai][x], j = g_cart_pair[LB][bi][x];
          const double* E = s_E[x];
          const auto sv = [&](int ii, int jj) { return E[(ii * EJ + jj) * MT]; };
          const auto tv = [&](int ii, int jj) {
            double r = -2.0 * be * be * sv(ii, jj + 2) + be * (2 * jj + 1) * sv(ii, jj);
            if (jj >= 2) r -= 0.5 * jj * (jj - 1) * sv(ii, jj - 2);
            return r;
          };
          s1[x] = sv(i, j);
          t1[x] = tv(i, j);
          ds[x] = 2.0 * al * sv(i + 1, j) - (i > 0 ? i * sv(i - 1, j) : 0.0);
          dt[x] = 2.0 * al * tv(i + 1, j) - (i > 0 ? i * tv(i - 1, j) : 0.0);
        }
#pragma unroll
        for (int x = 0; x < 3; ++x) {
          const int y = (x + 1) % 3, z = (x + 2) % 3;
          const double dS = s0 * ds[x] * s1[y] * s1[z];
          const double dT = s0 * (dt[x] * s1[y] * s1[z] + ds[x] * t1[y] * s1[z] + ds[x] * s1[y] * t1[z]);
          gS[0][x] += s_w[0][o] * dT - s_w[1][o] * dS;
#pragma unroll
          for (int k = 1; k < 4; ++k) gS[k][x] -= s_w[1 + k][o] * dS;
        }
      }
      // N[h] and its three X derivatives
      for (int h = lane; h < NH; h += 64) {
        const int tuv = s_h[h];
        const int t3[3] = {tuv & 15, (tuv >> 4) & 15, tuv >> 8};
        double n[4] = {0.0, 0.0, 0.0, 0.0};
        for (int o = 0; o < NO; ++o) {
          const int ai = o / NB, bi = o % NB;
          double e[3], d[3];
#pragma unroll
          for (int x = 0; x < 3; ++x) {
            const int i = g_cart_pair[LA][ai][x], j = g_cart_pair[LB][bi][x], t = t3[x];
            const double* E = s_E[x];
            e[x] = t <= i + j ? E[(i * EJ + j) * MT + t] : 0.0;
            double y = 2.0 * al * E[((i + 1) * EJ + j) * MT + t];
            if (i > 0) y -= i * E[((i - 1) * EJ + j) * MT + t];
            if (t > 0) y -= al * ip * E[(i * EJ + j) * MT + t - 1];
            d[x] = t <= i + j ? y : 0.0;
          }
          const double w = s_w[0][o];
          n[0] += w * e[0] * e[1] * e[2];
          n[1] += w * d[0] * e[1] * e[2];
          n[2] += w * e[0] * d[1] * e[2];
          n[3] += w * e[0] * e[1] * d[2];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) s_N[k][h] = n[k];
      }
      __syncthreads();
      const double Px = (al * xa[0] + be * xb[0]) * ip, Py = (al * xa[1] + be * xb[1]) * ip,
                   Pz = (al * xa[2] + be * xb[2]) * ip;
      for (int c0 = 0; c0 < natm; c0 += 16) {
        nuclear_r<L>(c0, natm, atm, cab * 2.0 * kPi * ip, p, Px, Py, Pz, boys, s_R);
        double F[3] = {0.0, 0.0, 0.0}, Q[3] = {0.0, 0.0, 0.0};
#pragma unroll 2
        for (int q = 0; q < HQ; ++q) {
          const int h = 4 * q + sub;
          if (h < NH) {
            const int tuv = s_h[h], t = tuv & 15, u = (tuv >> 4) & 15, v = tuv >> 8;
            const int r = u + v, s = t + r + 1;
            const double r0 = s_R[h * 16 + ax];
            const int b = s * (s + 1) * (s + 2) / 6 + r * (r + 1) / 2 + v;    // h + x; then h + y, h + z
            const double n0 = s_N[0][h];
            F[0] += n0 * s_R[b * 16 + ax];
            F[1] += n0 * s_R[(b + r + 1) * 16 + ax];
            F[2] += n0 * s_R[(b + r + 2) * 16 + ax];
#pragma unroll
            for (int e = 0; e < 3; ++e) Q[e] += s_N[1 + e][h] * r0;
          }
        }
#pragma unroll
        for (int e = 0; e < 3; ++e) {
          gA[e] += al * ip * F[e] + Q[e];
          gB[e] += be * ip * F[e] - Q[e];
          double c = F[e] + __shfl_xor(F[e], 16);
          c += __shfl_xor(c, 32);
          if (sub == 0 && c0 + ax < natm) atomicAdd(&grad[3 * (c0 + ax) + e], -f * c);
        }
      }
    }
  const int at_a = atom_a[ia], at_b = atom_a[ib];
#pragma unroll
  for (int e = 0; e < 3; ++e) {
    double v[6] = {gA[e] + gS[0][e], gB[e] - gS[0][e], gS[1][e], gS[2][e], gS[3][e], 0.0};
#pragma unroll
    for (int k = 0; k < 5; ++k)
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) v[k] += __shfl_xor(v[k], o);
    if (lane == 0) {
      atomicAdd(&grad[3 * at_a + e], f * v[0]);
      atomicAdd(&grad[3 * at_b + e], f * v[1]);
      if (at_a != at_b)
        for (int k = 1; k < 4; ++k) {
          atomicAdd(&grad[k * part + 3 * at_a + e], f * v[1 + k]);
          atomicAdd(&grad[k * part + 3 * at_b + e], -f * v[1 + k]);
        }
    }
  }
}

}  // namespace

void upload_int1e_tables(const C2SList& h, const int (&cart)[7][28][3]) {
  (void)hipMemcpyToSymbol(HIP_SYMBOL(g_c2s_pair), &h, sizeof(h));
  (void)hipMemcpyToSymbol(HIP_SYMBOL(g_cart_pair), cart, sizeof(cart));
}

#define DFKS_1E_CLASSES(X) X(0, 0) X(1, 0) X(1, 1) X(2, 0) X(2, 1) X(2, 2) X(3, 0) X(3, 1) X(3, 2) X(3, 3)
#define DFKS_1E_CLASSES_G(X) X(4, 0) X(4, 1) X(4, 2) X(4, 3) X(4, 4)   // a span's overlap alone

// S, T and V of one class of shell pairs (la >= lb, each unordered pair once), both triangles; natm = 0: V = 0
hipError_t launch_int1e(int la, int lb, const int2* pairs, int npair, const ShellSet& A, int natm, const double* atm,
                        const double* boys, double* S, double* T, double* V, int64_t nao, hipStream_t st) {
  if (npair == 0) return hipSuccess;
#define DFKS_1E(a, b) \
  if (la == a && lb == b) { \
    hipLaunchKernelGGL((k_int1e<a, b>), dim3((unsigned)npair), dim3(64), 0, st, pairs, A, natm, atm, boys, S, T, V, \
                       nao); \
    return hipGetLastError(); \
  }
  DFKS_1E_CLASSES(DFKS_1E)
  DFKS_1E_CLASSES_G(DFKS_1E)
#undef DFKS_1E
  return hipErrorInvalidValue;
}

hipError_t launch_int1e_grad(int la, int lb, const int2* pairs, int npair, const ShellSet& A, const int32_t* atom_a,
                             int natm, const double* atm, const double* boys, const double* P,
                             const double* const (&W)[4], int64_t nao, double* grad, int64_t part, hipStream_t st) {
  if (npair == 0) return hipSuccess;
  const Int1eW w{{W[0], W[1], W[2], W[3]}};
#define DFKS_1E(a, b) \
  if (la == a && lb == b) { \
    hipLaunchKernelGGL((k_int1e_pgrad<a, b>), dim3((unsigned)npair), dim3(64), 0, st, pairs, A, atom_a, natm, atm, \
                       boys, P, w, nao, grad, part); \
    return hipGetLastError(); \
  }
  DFKS_1E_CLASSES(DFKS_1E)
#undef DFKS_1E
  return hipErrorInvalidValue;
}

}  // namespace dfks
