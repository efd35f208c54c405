// Nuclear derivatives of the two- and three-centre integrals contracted with their densities, by bra
// pair: one workgroup per bra shell pair (and part of the auxiliary shells of one l_c), one template
// instance per class.
//
// With H and G of eri_pair.hip, sum_{AB,Cm} Gamma[AB][Cm] (AB|Cm) = sum_h N[h][Cm] G[h][Cm],
// N = H^T Gamma. The integral depends on the centres through P (in G) and through X = A - B (in H):
//   d/dP_x  sends G_h to G_{h + x} (one Hermite order up), d/dX_x replaces H by dH/dX, per axis
//   dE^{ij}_t / dX = 2a E^{i+1,j}_t - i E^{i-1,j}_t - (a/p) E^{ij}_{t-1};
//   d/dA = (a/p) d/dP + d/dX,  d/dB = (b/p) d/dP - d/dX,  d/dC = -d/dP.
// So four tables (H and its three X derivatives) multiply the same Gamma on
// v_mfma_f64_16x16x4f64 (rows = h, k = AB functions, columns = 16 auxiliary shells), and each lane
// weights its rows of the products with G and its three shifts from R in LDS: no derivative of a
// single integral is formed. Auxiliary centres collect in LDS per atom and go out once a workgroup.
// Bound by the matrix work (4 times the integrals') and the reads of R. A tree of 6 heavy atoms,
// def2-SVP: 6.6 ms for the Coulomb and the exchange term, 71 ms with a wavefront per task that
// differentiated each integral (k_eri_grad in eri.hip, kept for cartesian spans with l >= 2 and for
// more atoms than the LDS sums hold).
// One wavefront a SIMD has registers for all but the widest classes: spilled words (3,3,4) 450, (3,3,3) 275, (3,2,4)
// 199, (3,3,2) 104, (2,2,4) 102, (3,2,3) 85, (3,1,4) 68, (2,2,3) 7.
// Reference: dftax/ks/forces.py:128-270 (jax.grad through eri3c_bucketed.py:290-426).
#include <algorithm>
#include <cstdint>

#include "eri_pair.h"

namespace dfks {

namespace {

template <int LA, int LB, int LC>
struct GradCls {
  static constexpr int L = LA + LB + LC + 1, LAB = LA + LB;
  static constexpr int FB = nsph(LB), NM = nsph(LC), ROWS = nsph(LA) * FB;
  static constexpr int NH = n_tet(LAB), HT = (NH + 15) / 16, KQ = (ROWS + 3) / 4;
  static constexpr int R0 = LC > 0 ? n_tet(LC - 1) : 0, NR = n_tet(L) - R0;
  static constexpr int TSZ = HT * KQ * 64;                         // one table of one primitive pair
  static constexpr int NTAB = 4 * TSZ <= 8192 ? 4 : 1;             // tables held at a time
  static constexpr int ESZ = 3 * (LA + 2) * (LB + 1) * (LAB + 2);  // E up to (LA + 1, LB)
  static constexpr int NPC = NTAB * TSZ > 1280 ? 1 : (2560 / (NTAB * TSZ) > 24 ? 24 : 2560 / (NTAB * TSZ));
  static constexpr int NW = NR * 16 > 2600 ? 2 : 4;
};

// The tables tab0 .. tab0 + NTAB - 1 (0: H, 1..3: dH/dX_x) of the primitive pairs q0 .. q0 + n - 1, in the
// order of the MFMA A operand: [table][tile of 16 h][k / 4][lane], h = 16 tile + lane % 16, k = AB row
template <int LA, int LB, int LC>
__device__ __forceinline__ void grad_tables(const BraPair& b, int q0, int n, int tab0, int tid,
                                            double* __restrict__ s_T, double* __restrict__ s_E, double (*s_P)[6],
                                            double* __restrict__ s_f) {
  using K = GradCls<LA, LB, LC>;
  constexpr int NT = K::NW * 64, LAB = K::LAB, MT = LAB + 2, ES = K::ESZ / 3;
  for (int w = tid; w < 3 * n; w += NT) {
    const int q = w / 3, x = w - 3 * q;
    const int pa = (q0 + q) / b.npb, pb = (q0 + q) % b.npb;
    const double al = b.ea[pa], be = b.eb[pb];
    const double p = al + be, ip = 1.0 / p;
    const double ca = b.xa[x], cb = b.xb[x], ab = ca - cb;
    e_axis<LA + 1, LB>(-be * ab * ip, al * ab * ip, 0.5 * ip, s_E + q * K::ESZ + x * ES);
    s_P[q][x] = (al * ca + be * cb) * ip;
    if (x == 0) {
      const double dx = b.xa[0] - b.xb[0], dy = b.xa[1] - b.xb[1], dz = b.xa[2] - b.xb[2];
      s_P[q][3] = p;
      s_P[q][4] = al;
      s_P[q][5] = be;
      s_f[q] = b.ca[pa] * b.cb[pb] * exp(-al * be * ip * (dx * dx + dy * dy + dz * dz));
    }
  }
  __syncthreads();
  for (int w = tid; w < n * K::TSZ; w += NT) {
    const int q = w / K::TSZ, rem = w - q * K::TSZ, l = rem & 63;
    const int h = (rem / (K::KQ * 64)) * 16 + (l & 15), row = ((rem / 64) % K::KQ) * 4 + (l >> 4);
    double sum[4] = {0.0, 0.0, 0.0, 0.0};
    if (row < K::ROWS && h < K::NH) {
      int s = 0;
      while (h >= n_tet(s)) ++s;
      const int k = h - (s > 0 ? n_tet(s - 1) : 0);
      int r = 0;
      while (k >= (r + 1) * (r + 2) / 2) ++r;
      const int v = k - r * (r + 1) / 2;
      const int tuv[3] = {s - r, r - v, v};
      const int Ai = row / K::FB, Bi = row % K::FB;
      const int nA = LA >= 2 ? g_c2s_pair.n[LA][Ai] : 1, nB = LB >= 2 ? g_c2s_pair.n[LB][Bi] : 1;
      const double* E = s_E + q * K::ESZ;
      const double al = s_P[q][4], ap = al / s_P[q][3];
      for (int xa = 0; xa < nA; ++xa) {
        const int ai = LA >= 2 ? g_c2s_pair.cart[LA][Ai][xa] : Ai;
        const double wa = LA >= 2 ? g_c2s_pair.coef[LA][Ai][xa] : 1.0;
        for (int xb = 0; xb < nB; ++xb) {
          const int bi = LB >= 2 ? g_c2s_pair.cart[LB][Bi][xb] : Bi;
          const double wb = LB >= 2 ? wa * g_c2s_pair.coef[LB][Bi][xb] : wa;
          double e[3], d[3];
#pragma unroll
          for (int x = 0; x < 3; ++x) {
            const int i = g_cart_pair[LA][ai][x], j = g_cart_pair[LB][bi][x], t = tuv[x];
            const double* Ex = E + x * ES;
            e[x] = Ex[(i * (LB + 1) + j) * MT + t];
            double y = 2.0 * al * Ex[((i + 1) * (LB + 1) + j) * MT + t];
            if (i > 0) y -= i * Ex[((i - 1) * (LB + 1) + j) * MT + t];
            if (t > 0) y -= ap * Ex[(i * (LB + 1) + j) * MT + t - 1];
            d[x] = t <= i + j ? y : 0.0;    // above, the terms cancel
          }
          sum[0] += wb * e[0] * e[1] * e[2];
          sum[1] += wb * d[0] * e[1] * e[2];
          sum[2] += wb * e[0] * d[1] * e[2];
          sum[3] += wb * e[0] * e[1] * d[2];
        }
      }
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
      if (t >= tab0 && t < tab0 + K::NTAB) s_T[(q * K::NTAB + t - tab0) * K::TSZ + rem] = sum[t] * s_f[q];
  }
  __syncthreads();
}

template <int LA, int LB, int LC>
__global__ __launch_bounds__((GradCls<LA, LB, LC>::NW * 64)) void k_eri_pair_grad(
    const int2* __restrict__ pairs, const int32_t* __restrict__ aux, int naux_l, ShellSet A, ShellSet C,
    const int32_t* __restrict__ atom_a, const int32_t* __restrict__ atom_c, int natom,
    const double* __restrict__ boys, const double* __restrict__ Gm, int64_t gc, int64_t ga, int64_t gb,
    double* __restrict__ grad, int gper, int unit) {
  using K = GradCls<LA, LB, LC>;
  constexpr int L = K::L, FB = K::FB, NM = K::NM, HT = K::HT, KQ = K::KQ, NT = K::NW * 64;
  extern __shared__ double s_at[];      // [natom][3]: auxiliary centres
  __shared__ double s_T[K::NPC * K::NTAB * K::TSZ];
  __shared__ double s_E[K::NPC * K::ESZ];
  __shared__ double s_P[K::NPC][6];     // P, p, a, b
  __shared__ double s_f[K::NPC];
  __shared__ int s_tab[HT * 16];        // Hermite index h: base of its run in R (low 16 bits) and u + v
  __shared__ double s_R[K::NW][K::NR * 16];
  __shared__ double s_red[K::NW][6];

  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int ax = lane & 15, sub = lane >> 4;
  const int2 pr = pairs[blockIdx.x];
  const int ia = pr.x, ib = pr.y;
  const BraPair bp = bra_pair(A, ia, ib, unit != 0);
  const int npp = A.nprim[ia] * bp.npb;
  const int64_t ao_a = A.ao0[ia], ao_b = unit ? 0 : A.ao0[ib];

  for (int i = tid; i < 3 * natom; i += NT) s_at[i] = 0.0;
  for (int h = tid; h < HT * 16; h += NT) {
    int s = 0, e = h < K::NH ? h : 0;
    while (e >= n_tet(s)) ++s;
    const int k = e - (s > 0 ? n_tet(s - 1) : 0);
    int r = 0;
    while (k >= (r + 1) * (r + 2) / 2) ++r;
    const int v = k - r * (r + 1) / 2, sl = s + LC;
    s_tab[h] = (sl * (sl + 1) * (sl + 2) / 6 + r * (r + 1) / 2 + v - K::R0) | (r << 16) | (sl << 24);
  }

  double gA[3] = {0, 0, 0}, gB[3] = {0, 0, 0};
  const int ngrp = (naux_l + 15) / 16;
  const int gbeg = blockIdx.y * gper, gend = min(ngrp, gbeg + gper);
  double* Rw = s_R[wv] + ax;
  const bool one = npp <= K::NPC;
#pragma unroll 1
  for (int tab0 = 0; tab0 < 4; tab0 += K::NTAB) {
    if (one) grad_tables<LA, LB, LC>(bp, 0, npp, tab0, tid, s_T, s_E, s_P, s_f);
    for (int g0 = gbeg; g0 < gend; g0 += K::NW) {
      const int g = g0 + wv;
      const bool live = g < gend;          // uniform over the wavefront
      const int j = g * 16 + ax;
      const bool have = live && j < naux_l;
      const int ic = aux[have ? j : 0];
      const double Cx = C.centre[3 * ic], Cy = C.centre[3 * ic + 1], Cz = C.centre[3 * ic + 2];
      const int npc = C.nprim[ic], p0c = C.prim0[ic];
      const double* Gc = Gm + (int64_t)C.ao0[ic] * gc + ao_a * ga + ao_b * gb;
      int npcm = npc;
#pragma unroll
      for (int o = 1; o < 16; o <<= 1) npcm = max(npcm, __shfl_xor(npcm, o));
      double sc[3] = {0, 0, 0};            // d/dP of this lane's auxiliary shell
      for (int q0 = 0; q0 < npp; q0 += K::NPC) {
        const int nq = min(K::NPC, npp - q0);
        if (!one) {
          __syncthreads();
          grad_tables<LA, LB, LC>(bp, q0, nq, tab0, tid, s_T, s_E, s_P, s_f);
        }
        if (!live) continue;
        for (int q = 0; q < nq; ++q) {
          const double p = s_P[q][3];
          const double x = s_P[q][0] - Cx, y = s_P[q][1] - Cy, z = s_P[q][2] - Cz;
          double sp[3] = {0, 0, 0}, sx[3] = {0, 0, 0};
          for (int pc = 0; pc < npcm; ++pc) {
            const int pi = p0c + (pc < npc ? pc : 0);
            const double gam = C.exps[pi];
            const double cc = have && pc < npc ? C.coefs[pi] : 0.0;
            const double rho = p * gam / (p + gam);
            double pref = cc * 2.0 * 17.493418327624862 / (p * gam * sqrt(p + gam));  // 2 pi^2.5
            const double i2g = -0.5 / gam;
#pragma unroll
            for (int k = 0; k < LC; ++k) pref *= i2g;
            double Zc[L + 1], Zp[L + 1];
            boys_op<L>(rho * (x * x + y * y + z * z), rho, C.omega, Zc, boys);
            const double n2r = -2.0 * rho;
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
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // the last reads of R are done
            r_planes<L, LC, K::R0, 0>(x, y, z, sub, Zc, Zp, Rw);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            const double* Tq = s_T + q * K::NTAB * K::TSZ + lane;
#pragma unroll
            for (int m = 0; m < NM; ++m) {
              __builtin_amdgcn_sched_barrier(0);   // one m at a time: its registers are enough for a wavefront
              double gm[KQ];
#pragma unroll
              for (int kq = 0; kq < KQ; ++kq) {
                const int row = min(4 * kq + sub, K::ROWS - 1);     // rows past the last meet zeros
                gm[kq] = Gc[m * gc + (row / FB) * ga + (row % FB) * gb];
              }
#pragma unroll 1
              for (int ht = 0; ht < HT; ++ht) {
                dbl4 acc[K::NTAB];
#pragma unroll
                for (int t = 0; t < K::NTAB; ++t) acc[t] = dbl4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int kq = 0; kq < KQ; ++kq)
#pragma unroll
                  for (int t = 0; t < K::NTAB; ++t)
                    acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(Tq[t * K::TSZ + (ht * KQ + kq) * 64], gm[kq],
                                                                  acc[t], 0, 0, 0);
                // result register i: Hermite index 16 ht + sub + 4 i, auxiliary shell ax
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                  const int tb = s_tab[16 * ht + sub + 4 * i];
                  const int r = (tb >> 16) & 0xff, sl = tb >> 24, b0 = tb & 0xffff;
                  const int bx = b0 + (sl + 1) * (sl + 2) / 2;     // one order up: h + x, then h + y, h + z
                  double G[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                  for (int d = 0; d <= LC; ++d)
#pragma unroll
                    for (int zz = 0; zz <= d; ++zz) {
                      const double cf = c2s_coef<LC>(d * (d + 1) / 2 + zz, m);
                      if (cf != 0.0) {
                        const int o = d * (d + 1) / 2 + zz;
                        G[0] += cf * Rw[(b0 + d * r + o) * 16];
                        G[1] += cf * Rw[(bx + d * r + o) * 16];
                        const int by = bx + r + 1 + d * (r + 1) + o;
                        G[2] += cf * Rw[by * 16];
                        G[3] += cf * Rw[(by + 1) * 16];
                      }
                    }
                  if constexpr (K::NTAB == 4) {
#pragma unroll
                    for (int e = 0; e < 3; ++e) {
                      sp[e] += acc[0][i] * G[1 + e];
                      sx[e] += acc[1 + e][i] * G[0];
                    }
                  } else if (tab0 == 0) {
#pragma unroll
                    for (int e = 0; e < 3; ++e) sp[e] += acc[0][i] * G[1 + e];
                  } else {
#pragma unroll
                    for (int e = 0; e < 3; ++e) sx[e] += tab0 == e + 1 ? acc[0][i] * G[0] : 0.0;
                  }
                }
              }
            }
          }
          const double fa = s_P[q][4] / p, fb = s_P[q][5] / p;
#pragma unroll
          for (int e = 0; e < 3; ++e) {
            gA[e] += fa * sp[e] + sx[e];
            gB[e] += fb * sp[e] - sx[e];
            sc[e] += sp[e];
          }
        }
      }
      // the shell's four lanes, then its atom
#pragma unroll
      for (int e = 0; e < 3; ++e) {
        sc[e] += __shfl_xor(sc[e], 16);
        sc[e] += __shfl_xor(sc[e], 32);
      }
      if (have && sub == 0 && tab0 == 0) {
        const int at = atom_c[ic];
#pragma unroll
        for (int e = 0; e < 3; ++e) atomicAdd(&s_at[3 * at + e], -sc[e]);
      }
    }
    if (K::NTAB < 4) __syncthreads();   // the next table overwrites this one
  }
  const double f = !unit && ia != ib ? 2.0 : 1.0;
#pragma unroll
  for (int e = 0; e < 3; ++e) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      gA[e] += __shfl_xor(gA[e], o);
      gB[e] += __shfl_xor(gB[e], o);
    }
    if (lane == 0) {
      s_red[wv][e] = gA[e];
      s_red[wv][3 + e] = gB[e];
    }
  }
  __syncthreads();
  if (tid < 6 && (tid < 3 || !unit)) {
    double t = 0.0;
    for (int w = 0; w < K::NW; ++w) t += s_red[w][tid];
    atomicAdd(&grad[3 * atom_a[tid < 3 ? ia : ib] + tid % 3], f * t);
  }
  for (int i = tid; i < 3 * natom; i += NT)
    if (s_at[i] != 0.0) atomicAdd(&grad[i], f * s_at[i]);
}

template <int LA, int LB, int LC>
hipError_t go_grad(const int2* pairs, int npair, const int32_t* aux, int naux_l, const ShellSet& A, const ShellSet& C,
                   const int32_t* atom_a, const int32_t* atom_c, int natom, const double* boys, const double* G,
                   int64_t gc, int64_t ga, int64_t gb, double* grad, int unit, hipStream_t st) {
  using K = GradCls<LA, LB, LC>;
  const int ngrp = (naux_l + 15) / 16;
  const int nseg = std::max(1, std::min((ngrp + K::NW - 1) / K::NW, 1024 / npair));
  int gper = (ngrp + nseg - 1) / nseg;
  gper = (gper + K::NW - 1) / K::NW * K::NW;
  const dim3 grid((unsigned)npair, (unsigned)((ngrp + gper - 1) / gper));
  hipLaunchKernelGGL((k_eri_pair_grad<LA, LB, LC>), grid, dim3(K::NW * 64), 3 * natom * sizeof(double), st, pairs, aux,
                     naux_l, A, C, atom_a, atom_c, natom, boys, G, gc, ga, gb, grad, gper, unit);
  return hipGetLastError();
}

}  // namespace

void upload_pair_grad_tables(const C2SList& h, const int (&cart)[7][28][3]) {
  (void)hipMemcpyToSymbol(HIP_SYMBOL(g_c2s_pair), &h, sizeof(h));
  (void)hipMemcpyToSymbol(HIP_SYMBOL(g_cart_pair), cart, sizeof(cart));
}

// atoms whose sums fit beside the tables in LDS
constexpr int kGradMaxAtoms = 1024;

// Whether the class and the spans go through the bra-pair kernel (else launch_eri_grad).
bool eri_pair_grad_has(int la, const ShellSet& A, const ShellSet& C, int natom, int unit) {
  return C.spherical && (A.spherical || la < 2) && natom <= kGradMaxAtoms && (unit ? la <= 4 : la <= 3);
}

// grad[atom] += sum Gamma d(ab|c)/dR over the class's pairs (la >= lb, ia >= ib, off-diagonal pairs twice) and
// auxiliary shells; Gamma[c gc + a ga + b gb]. unit: two-centre, pairs (shell, shell), lb = 0.
hipError_t launch_eri_pair_grad(int la, int lb, int lc, const int2* pairs, int npair, const int32_t* aux, int naux_l,
                                const ShellSet& A, const ShellSet& C, const int32_t* atom_a, const int32_t* atom_c,
                                int natom, int unit, const double* boys, const double* G, int64_t gc, int64_t ga,
                                int64_t gb, double* grad, hipStream_t st) {
  if (npair == 0 || naux_l == 0) return hipSuccess;
  if (!eri_pair_grad_has(la, A, C, natom, unit) || (unit && lb != 0)) return hipErrorInvalidValue;
#define DFKS_GRAD(a, b) \
  if (la == a && lb == b) { \
    switch (lc) { \
      case 0: return go_grad<a, b, 0>(pairs, npair, aux, naux_l, A, C, atom_a, atom_c, natom, boys, G, gc, ga, gb, grad, unit, st); \
      case 1: return go_grad<a, b, 1>(pairs, npair, aux, naux_l, A, C, atom_a, atom_c, natom, boys, G, gc, ga, gb, grad, unit, st); \
      case 2: return go_grad<a, b, 2>(pairs, npair, aux, naux_l, A, C, atom_a, atom_c, natom, boys, G, gc, ga, gb, grad, unit, st); \
      case 3: return go_grad<a, b, 3>(pairs, npair, aux, naux_l, A, C, atom_a, atom_c, natom, boys, G, gc, ga, gb, grad, unit, st); \
      case 4: return go_grad<a, b, 4>(pairs, npair, aux, naux_l, A, C, atom_a, atom_c, natom, boys, G, gc, ga, gb, grad, unit, st); \
      default: return hipErrorInvalidValue; \
    } \
  }
  DFKS_GRAD(0, 0) DFKS_GRAD(1, 0) DFKS_GRAD(1, 1) DFKS_GRAD(2, 0) DFKS_GRAD(2, 1) DFKS_GRAD(2, 2)
  DFKS_GRAD(3, 0) DFKS_GRAD(3, 1) DFKS_GRAD(3, 2) DFKS_GRAD(3, 3) DFKS_GRAD(4, 0)
#undef DFKS_GRAD
  return hipErrorInvalidValue;
}

}  // namespace dfks
