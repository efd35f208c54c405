// Three-centre (ab|c) with a spherical auxiliary span, by bra pair: one
// workgroup per bra shell pair (and a segment of the auxiliary shells of one
// l_c), one template instance per class.
//
// McMurchie-Davidson (dftax/integrals/eri3c_bucketed.py:290-426) arranged as a
// matrix product per bra primitive pair:
//   (AB|C m) += sum_h H[AB][h] G[h][m],   h = (t,u,v), t+u+v <= l_a + l_b
//   H[AB][h]  = c_a c_b K_AB sum_cart c2s_a c2s_b E_t E_u E_v    (bra only)
//   G[h][m]   = pref (-1)^l_c (2 gamma)^-l_c sum_xyz c2s_c[xyz][m] R_{t+x,u+y,v+z}
// The auxiliary side has no Hermite expansion: a real solid harmonic times a
// Gaussian is (2 gamma)^-l S_lm(d/dC) of the plain Gaussian (Hobson's theorem;
// the lower terms of the single-centre expansion cancel because S_lm is
// harmonic), so only R of total order l_c and above enters.
//
// Layout: a wavefront takes 16 auxiliary shells at a time, 4 lanes a shell.
//  - H is formed once per workgroup in LDS and read as the A operand of
//    v_mfma_f64_16x16x4f64 (rows = AB functions, k = Hermite index); every
//    auxiliary shell of the segment reuses it.
//  - R: entries of one v form a (t,u) triangle whose ladder needs only
//    R^(n)_00v, so the 4 lanes of a shell take v = 4k + lane/16 and run the
//    triangle's ladder in registers, then store it to LDS once. No table
//    lookups and no workgroup barriers.
//  - G is formed by the lane that holds it as the B operand (k = lane/16, n =
//    auxiliary shell), from l_c+1 runs of R at fixed offsets: in the order
//    t+u+v the entry (t+x, u+y, v+z) sits at base + (y+z)(u+v) + const.
// Bound by FP64 matrix work in the d and f classes and by the Boys function
// and R in the low ones. One workgroup walks all auxiliary shells of its class
// (the segments only give small molecules enough workgroups), so H is paid
// once. The 31 classes of l_a + l_b + l_c >= 4 of (H2O)_24 def2-TZVP take
// 15.7 ms on the MI355X against 241 ms with a wavefront per task (lane 0 alone
// on the Boys function, table lookups in the ladder); (fp|d) 0.93 against 15.9
// ms, (ff|g) 0.23 against 6.3 ms.
#include <algorithm>
#include <cstdint>

#include "eri_pair.h"

namespace dfks {

namespace {

// A class's sizes: AB rows and Hermite indices padded to the MFMA shape, R entries of order >= LC
template <int LA, int LB, int LC>
struct PairCls {
  static constexpr int L = LA + LB + LC, LAB = LA + LB;
  static constexpr int FA = nsph(LA), FB = nsph(LB), NM = nsph(LC), ROWS = FA * FB;
  static constexpr int MTA = (ROWS + 15) / 16, NH = n_tet(LAB), KQ = (NH + 3) / 4;
  // row tiles of one workgroup: half of them where all would not leave registers for R
  static constexpr int PARTS = MTA * NM > 24 ? 2 : 1, MT = (MTA + PARTS - 1) / PARTS;
  static constexpr int R0 = LC > 0 ? n_tet(LC - 1) : 0, NR = n_tet(L) - R0;
  static constexpr int HSZ = MT * KQ * 64;                       // doubles of H per primitive pair
  static constexpr int ESZ = 3 * (LA + 1) * (LB + 1) * (LAB + 1);  // doubles of E per primitive pair
  // primitive pairs whose H is held at a time (18 KB where it is more than one), wavefronts per workgroup
  static constexpr int NPC = HSZ > 2304 ? 1 : (2304 / HSZ > 36 ? 36 : 2304 / HSZ);
  static constexpr int NW = NR * 16 > 2600 ? 2 : 4;
  // wavefronts a SIMD. With two the accumulators, R's ladder and G do not all fit in (3,2,1), which spills 56 words,
  // (2,1,4) 29, (3,0,4) 25, (3,1,2) 16, (2,2,2) 12, and 2 in (3,2,0) and the two-centre (4,0,3)
  static constexpr int OCC = MT * NM * 8 > 80 ? 1 : 2;
};

// H (rows row0 ..), P and p of the primitive pairs q0 .. q0 + n - 1 into LDS, by the whole workgroup
template <int LA, int LB, int LC>
__device__ __forceinline__ void bra_tables(const BraPair& b, int q0, int n, int row0, int tid, double* __restrict__ s_H,
                                           double* __restrict__ s_E, double (*s_P)[4], double* __restrict__ s_f) {
  using K = PairCls<LA, LB, LC>;
  constexpr int LAB = K::LAB, FB = K::FB, KQ = K::KQ, NH = K::NH, NT = K::NW * 64, ES = K::ESZ / 3;
  for (int w = tid; w < 3 * n; w += NT) {
    const int q = w / 3, x = w - 3 * q;
    const int pa = (q0 + q) / b.npb, pb = (q0 + q) % b.npb;
    const double al = b.ea[pa], be = b.eb[pb];
    const double p = al + be, ip = 1.0 / p;
    const double ca = b.xa[x], cb = b.xb[x], ab = ca - cb;
    e_axis<LA, LB>(-be * ab * ip, al * ab * ip, 0.5 * ip, s_E + q * K::ESZ + x * ES);
    s_P[q][x] = (al * ca + be * cb) * ip;
    if (x == 0) {
      const double dx = b.xa[0] - b.xb[0], dy = b.xa[1] - b.xb[1], dz = b.xa[2] - b.xb[2];
      s_P[q][3] = p;
      s_f[q] = b.ca[pa] * b.cb[pb] * exp(-al * be * ip * (dx * dx + dy * dy + dz * dz));
    }
  }
  __syncthreads();
  for (int w = tid; w < n * K::HSZ; w += NT) {
    const int q = w / K::HSZ, rem = w - q * K::HSZ;
    const int row = row0 + (rem / (KQ * 64)) * 16 + (rem & 15), h = (rem % (KQ * 64)) >> 4;
    double sum = 0.0;
    if (row < K::ROWS && h < NH) {
      int s = 0;
      while (h >= n_tet(s)) ++s;
      const int k = h - (s > 0 ? n_tet(s - 1) : 0);
      int r = 0;
      while (k >= (r + 1) * (r + 2) / 2) ++r;
      const int v = k - r * (r + 1) / 2, u = r - v, t = s - r;
      const int Ai = row / FB, Bi = row % FB;
      const int nA = LA >= 2 ? g_c2s_pair.n[LA][Ai] : 1, nB = LB >= 2 ? g_c2s_pair.n[LB][Bi] : 1;
      const double* E = s_E + q * K::ESZ;
      for (int xa = 0; xa < nA; ++xa) {
        const int ai = LA >= 2 ? g_c2s_pair.cart[LA][Ai][xa] : Ai;
        const double wa = LA >= 2 ? g_c2s_pair.coef[LA][Ai][xa] : 1.0;
        const int a0 = g_cart_pair[LA][ai][0], a1 = g_cart_pair[LA][ai][1], a2 = g_cart_pair[LA][ai][2];
        for (int xb = 0; xb < nB; ++xb) {
          const int bi = LB >= 2 ? g_c2s_pair.cart[LB][Bi][xb] : Bi;
          const double wb = LB >= 2 ? wa * g_c2s_pair.coef[LB][Bi][xb] : wa;
          const int b0 = g_cart_pair[LB][bi][0], b1 = g_cart_pair[LB][bi][1], b2 = g_cart_pair[LB][bi][2];
          sum += wb * E[(a0 * (LB + 1) + b0) * (LAB + 1) + t] *
                 E[ES + (a1 * (LB + 1) + b1) * (LAB + 1) + u] *
                 E[2 * ES + (a2 * (LB + 1) + b2) * (LAB + 1) + v];
        }
      }
      sum *= s_f[q];
    }
    s_H[w] = sum;
  }
  __syncthreads();
}

template <int LA, int LB, int LC>
__global__ __launch_bounds__((PairCls<LA, LB, LC>::NW * 64), (PairCls<LA, LB, LC>::OCC)) void k_eri_pair(
    const int2* __restrict__ pairs, const int32_t* __restrict__ aux, int naux_l, ShellSet A, ShellSet C,
    const double* __restrict__ boys, double* __restrict__ out, int64_t sa, int64_t sb, int64_t c0, int tr,
    int gper, int unit) {
  using K = PairCls<LA, LB, LC>;
  constexpr int L = K::L, LAB = K::LAB, FA = K::FA, FB = K::FB, NM = K::NM, MT = K::MT, KQ = K::KQ, NH = K::NH;
  constexpr int NT = K::NW * 64;
  __shared__ double s_H[K::NPC * K::HSZ];
  __shared__ double s_E[K::NPC * K::ESZ];
  __shared__ double s_P[K::NPC][4];   // P and the exponent p
  __shared__ double s_f[K::NPC];      // c_a c_b K_AB
  __shared__ int s_tab[KQ * 4];       // Hermite index h: base of its R run (low 16 bits) and u + v
  __shared__ double s_R[K::NW][K::NR * 16];

  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int ax = lane & 15, sub = lane >> 4;
  const int2 pr = pairs[blockIdx.x];
  const int row0 = blockIdx.z * (MT * 16);   // first AB row of this workgroup's tiles
  const int ia = pr.x, ib = pr.y;
  const BraPair bp = bra_pair(A, ia, ib, unit != 0);
  const int npp = A.nprim[ia] * bp.npb;
  const int64_t ao_a = A.ao0[ia], ao_b = unit ? 0 : A.ao0[ib];

  for (int h = tid; h < KQ * 4; h += NT) {
    int s = 0, e = h < NH ? h : 0;
    while (e >= n_tet(s)) ++s;
    const int k = e - (s > 0 ? n_tet(s - 1) : 0);
    int r = 0;
    while (k >= (r + 1) * (r + 2) / 2) ++r;
    const int v = k - r * (r + 1) / 2;
    const int sl = s + LC;
    s_tab[h] = (sl * (sl + 1) * (sl + 2) / 6 + r * (r + 1) / 2 + v - K::R0) | (r << 16);
  }

  const bool one = npp <= K::NPC;
  if (one) bra_tables<LA, LB, LC>(bp, 0, npp, row0, tid, s_H, s_E, s_P, s_f);

  const int ngrp = (naux_l + 15) / 16;
  const int gbeg = blockIdx.y * gper, gend = min(ngrp, gbeg + gper);
  double* Rw = s_R[wv] + ax;
  for (int g0 = gbeg; g0 < gend; g0 += K::NW) {
    const int g = g0 + wv;
    const bool live = g < gend;          // uniform over the wavefront
    const int j = g * 16 + ax;
    const bool have = live && j < naux_l;
    const int ic = aux[have ? j : 0];
    const double Cx = C.centre[3 * ic], Cy = C.centre[3 * ic + 1], Cz = C.centre[3 * ic + 2];
    const int npc = C.nprim[ic], p0c = C.prim0[ic];
    int npcm = npc;                      // the longest contraction of the wavefront's shells
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) npcm = max(npcm, __shfl_xor(npcm, o));
    dbl4 acc[MT][NM];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int m = 0; m < NM; ++m) acc[mt][m] = dbl4{0.0, 0.0, 0.0, 0.0};

    for (int q0 = 0; q0 < npp; q0 += K::NPC) {
      const int nq = min(K::NPC, npp - q0);
      if (!one) {
        __syncthreads();                 // every wavefront is done with the previous chunk
        bra_tables<LA, LB, LC>(bp, q0, nq, row0, tid, s_H, s_E, s_P, s_f);
      }
      if (!live) continue;
      for (int q = 0; q < nq; ++q) {
        const double p = s_P[q][3];
        const double x = s_P[q][0] - Cx, y = s_P[q][1] - Cy, z = s_P[q][2] - Cz;
        for (int pc = 0; pc < npcm; ++pc) {
          const int pi = p0c + (pc < npc ? pc : 0);
          const double ga = C.exps[pi];
          const double cc = pc < npc ? C.coefs[pi] : 0.0;
          const double rho = p * ga / (p + ga);
          double pref = cc * 2.0 * 17.493418327624862 / (p * ga * sqrt(p + ga));  // 2 pi^2.5
          const double i2g = -0.5 / ga;  // (-1)^l_c (2 gamma)^-l_c
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
          // R^(n)_00v of this lane's first plane v = sub
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
          const double* Hq = s_H + q * K::HSZ + lane;
#pragma unroll 2
          for (int kq = 0; kq < KQ; ++kq) {
            const int tb = s_tab[4 * kq + sub];
            const int r = (tb >> 16) * 16;
            const double* Rb = Rw + (tb & 0xffff) * 16;
            double G[NM];
#pragma unroll
            for (int m = 0; m < NM; ++m) G[m] = 0.0;
#pragma unroll
            for (int d = 0; d <= LC; ++d) {
              const double* Rd = Rb + d * r;
#pragma unroll
              for (int zz = 0; zz <= d; ++zz) {
                const double rv = Rd[(d * (d + 1) / 2 + zz) * 16];
#pragma unroll
                for (int m = 0; m < NM; ++m) {
                  const double cf = c2s_coef<LC>(d * (d + 1) / 2 + zz, m);
                  if (cf != 0.0) G[m] += cf * rv;
                }
              }
            }
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
              const double a = Hq[(mt * KQ + kq) * 64];
#pragma unroll
              for (int m = 0; m < NM; ++m)
                acc[mt][m] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, G[m], acc[mt][m], 0, 0, 0);
            }
          }
        }
      }
    }
    if (have) {
      // result register i of lane (sub, ax): row sub + 4 i of the tile, auxiliary shell ax
      const int64_t ao_c = C.ao0[ic] - c0;
  #pragma unroll
      for (int mt = 0; mt < MT; ++mt)
  #pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int row = row0 + mt * 16 + sub + 4 * i;
          if (row < K::ROWS) {
            const int Ai = row / FB, Bi = row % FB;
            double* o1 = out + (ao_a + Ai) * sa + (ao_b + Bi) * sb + ao_c;
  #pragma unroll
            for (int m = 0; m < NM; ++m) o1[m] = acc[mt][m][i];
            if (tr && ia != ib) {
              double* o2 = out + (ao_b + Bi) * sa + (ao_a + Ai) * sb + ao_c;
  #pragma unroll
              for (int m = 0; m < NM; ++m) o2[m] = acc[mt][m][i];
            }
          }
        }
    }
  }
}

template <int LA, int LB, int LC>
hipError_t go_pair(const int2* pairs, int npair, const int32_t* aux, int naux_l, const ShellSet& A, const ShellSet& C,
                   const double* boys, double* out, int64_t sa, int64_t sb, int64_t c0, int tr, hipStream_t st,
                   int unit = 0) {
  using K = PairCls<LA, LB, LC>;
  const int ngrp = (naux_l + 15) / 16;
  // auxiliary segments: enough workgroups for the chip, at least one group per wavefront
  const int nseg = std::max(1, std::min((ngrp + K::NW - 1) / K::NW, 2048 / npair));
  int gper = (ngrp + nseg - 1) / nseg;
  gper = (gper + K::NW - 1) / K::NW * K::NW;
  const dim3 grid((unsigned)npair, (unsigned)((ngrp + gper - 1) / gper), (unsigned)K::PARTS);
  hipLaunchKernelGGL((k_eri_pair<LA, LB, LC>), grid, dim3(K::NW * 64), 0, st, pairs, aux, naux_l, A, C, boys, out, sa,
                     sb, c0, tr, gper, unit);
  return hipGetLastError();
}

}  // namespace

void upload_pair_tables(const C2SList& h, const int (&cart)[7][28][3]) {
  (void)hipMemcpyToSymbol(HIP_SYMBOL(g_c2s_pair), &h, sizeof(h));
  (void)hipMemcpyToSymbol(HIP_SYMBOL(g_cart_pair), cart, sizeof(cart));
}

// Every 3-centre class with l_b <= l_a <= 3, l_c <= 4; spherical auxiliary shells, and spherical
// orbital shells where l_a >= 2 (the caller checks both).
hipError_t launch_eri_pair(int la, int lb, int lc, const int2* pairs, int npair, const int32_t* aux, int naux_l,
                           const ShellSet& A, const ShellSet& C, const double* boys, double* out, int64_t sa,
                           int64_t sb, int64_t c0, int tr, hipStream_t st) {
  if (npair == 0 || naux_l == 0) return hipSuccess;
  if (!C.spherical || (la >= 2 && !A.spherical)) return hipErrorInvalidValue;
#define DFKS_PAIR(a, b) \
  if (la == a && lb == b) { \
    switch (lc) { \
      case 0: return go_pair<a, b, 0>(pairs, npair, aux, naux_l, A, C, boys, out, sa, sb, c0, tr, st); \
      case 1: return go_pair<a, b, 1>(pairs, npair, aux, naux_l, A, C, boys, out, sa, sb, c0, tr, st); \
      case 2: return go_pair<a, b, 2>(pairs, npair, aux, naux_l, A, C, boys, out, sa, sb, c0, tr, st); \
      case 3: return go_pair<a, b, 3>(pairs, npair, aux, naux_l, A, C, boys, out, sa, sb, c0, tr, st); \
      case 4: return go_pair<a, b, 4>(pairs, npair, aux, naux_l, A, C, boys, out, sa, sb, c0, tr, st); \
      default: return hipErrorInvalidValue; \
    } \
  }
  DFKS_PAIR(0, 0) DFKS_PAIR(1, 0) DFKS_PAIR(1, 1) DFKS_PAIR(2, 0) DFKS_PAIR(2, 1) DFKS_PAIR(2, 2)
  DFKS_PAIR(3, 0) DFKS_PAIR(3, 1) DFKS_PAIR(3, 2) DFKS_PAIR(3, 3)
#undef DFKS_PAIR
  return hipErrorInvalidValue;
}

// Two-centre (p|c), one class: p over the nshell shells of `pairs` (x: the shell), l_p <= 4, into
// out[p * sa + c]; spherical where l >= 2 (the caller checks).
hipError_t launch_eri2_pair(int la, int lc, const int2* pairs, int nshell, const int32_t* aux, int naux_l,
                            const ShellSet& A, const double* boys, double* out, int64_t sa, hipStream_t st) {
  if (nshell == 0 || naux_l == 0) return hipSuccess;
  if (!A.spherical) return hipErrorInvalidValue;
#define DFKS_PAIR2(a) \
  if (la == a) { \
    switch (lc) { \
      case 0: return go_pair<a, 0, 0>(pairs, nshell, aux, naux_l, A, A, boys, out, sa, 0, 0, 0, st, 1); \
      case 1: return go_pair<a, 0, 1>(pairs, nshell, aux, naux_l, A, A, boys, out, sa, 0, 0, 0, st, 1); \
      case 2: return go_pair<a, 0, 2>(pairs, nshell, aux, naux_l, A, A, boys, out, sa, 0, 0, 0, st, 1); \
      case 3: return go_pair<a, 0, 3>(pairs, nshell, aux, naux_l, A, A, boys, out, sa, 0, 0, 0, st, 1); \
      case 4: return go_pair<a, 0, 4>(pairs, nshell, aux, naux_l, A, A, boys, out, sa, 0, 0, 0, st, 1); \
      default: return hipErrorInvalidValue; \
    } \
  }
  DFKS_PAIR2(0) DFKS_PAIR2(1) DFKS_PAIR2(2) DFKS_PAIR2(3) DFKS_PAIR2(4)
#undef DFKS_PAIR2
  return hipErrorInvalidValue;
}

}  // namespace dfks
