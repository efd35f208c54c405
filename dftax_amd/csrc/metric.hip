// The factor of the fitting metric and the fitted tensor (FP64).
//
// V+ = L L^T over the eigenvectors of (P|Q) above cutoff * (largest eigenvalue). Where all of them are
// above it, any L with L L^T = V^-1 spans the same space, and L = C^-T from the Cholesky factor V = C C^T
// needs no eigenvectors. Whether all are above it is decided by two more factorisations that run in the
// same launches: V - cutoff t I and t I - V have Cholesky factors exactly when every eigenvalue lies
// strictly between cutoff t and t (t: a little more than the largest Ritz value of a short Lanczos run).
// If one of the three meets a pivot that is not positive, the caller takes the eigenvectors.
//
// (H2O)_8 def2-TZVP, 920 functions: 1.3 ms against 24 ms for the eigenvectors, a chain of several thousand
// small kernels; 2760 functions 11 ms. One eigenvalue at or under the cutoff costs the eigenvectors on top of the
// attempt, as for trees of about 12 heavy atoms and more (smallest eigenvalue 1e-7 of the largest at 10).
//
// Rounding: B B^T against 80 bits (norm against norm, 200 pairs; 35 geometries of water, (H2O)_4, (H2O)_8 and trees of
// 2 to 10 heavy atoms, condition 1e6 to 1e7) is off by 0.4 to 2.2e-15, 0.8e-15 in the geometric mean; with rocSOLVER's
// eigenvectors by 1.2 to 4.9e-15, 2.2e-15. That holds for fitting shells by falling l and exponent, the order in which
// the handle keeps them: taken atom by atom the factor's products with the integrals cancel more, 2.0 to 7.1e-15 on
// trees of 3 to 10 heavy atoms, and neither substitution instead of the blocks' inverses nor a refined panel mends that.
//
// Layout: one array of rows of ld = 64 ceil(n / 64) doubles, padded with a unit diagonal: V, the
// identity, and the two shifted matrices. A step takes 64 columns: their diagonal blocks are factored and
// inverted, one wavefront each with a row a lane in registers (k_chol_diag); the rows below, and the
// identity's rows down to the step's, are multiplied by the inverse (k_chol_panel); the columns to the
// right are updated (k_chol_update). All products are X Y^T with k along the rows of both, so their
// fragments load straight from global memory in 32-byte runs. The identity's rows end as C^-T.
// Bound by the chain of n / 64 steps (three launches and 64 pivots each).
#include <algorithm>
#include <cstdint>

#include "dfks_common.h"

namespace dfks {

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef double f64x2u __attribute__((ext_vector_type(2), aligned(8)));   // rows start on any 8 bytes

constexpr int kNB = 64;

// acc[i][j] += X Y^T over 64 k: X rows x0 + 16 i + li, Y rows y0 + 16 j + li (2 x 2 tiles of 16)
__device__ __forceinline__ void nt_32x32(const double* __restrict__ X, const double* __restrict__ Y, int64_t ldx,
                                         int64_t ldy, f64x4 (&acc)[2][2]) {
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const double *xr = X + li * ldx + 4 * lk, *yr = Y + li * ldy + 4 * lk;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    f64x4 x[2], y[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      x[i] = *reinterpret_cast<const f64x4*>(xr + 16 * i * ldx + 16 * q);
      y[i] = *reinterpret_cast<const f64x4*>(yr + 16 * i * ldy + 16 * q);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[i][s], y[j][s], acc[i][j], 0, 0, 0);
  }
}

// matrix z of the array: 0 V, then (after the identity) the shifted ones
__device__ __forceinline__ int64_t mat_off(int z, int64_t ld) { return (z == 0 ? 0 : z + 1) * ld * ld; }

__global__ __launch_bounds__(256) void k_chol_start(int n, int ld, const double* __restrict__ V, double cutoff,
                                                    double top, double* __restrict__ A, int* __restrict__ flag) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, nn = (int64_t)ld * ld;
  if (i == 0) *flag = 0;
  if (i >= nn) return;
  const int r = (int)(i / ld), c = (int)(i % ld);
  const bool in = r < n && c < n;
  const double v = in ? V[(int64_t)r * n + c] : 0.0, d = r == c ? 1.0 : 0.0;
  A[i] = in ? v : d;
  A[nn + i] = d;
  A[2 * nn + i] = in ? v - d * cutoff * top : d;
  A[3 * nn + i] = in ? d * top - v : d;
}

// Columns J.. of a diagonal block's factor, row `lane` of the block in r; 1 / l_jj to s_i. The row fills the
// registers, so the reads of a column are taken 16 at a time, used there, and not where the result is next needed.
template <int J>
__device__ __forceinline__ void chol_cols(int lane, double (&r)[kNB], double (*s_L)[kNB + 2], double* s_i, bool& bad) {
  if constexpr (J < kNB) {
    const double p = __shfl(r[J], J);
    bad = bad || !(p > 0.0);
    const double inv = 1.0 / sqrt(p), l = lane >= J ? r[J] * inv : 0.0;
    s_L[J][lane] = l;   // column J
    if (lane == J) s_i[J] = inv;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int c0 = 0; c0 < kNB; c0 += 16) {
      if (c0 + 15 > J) {
        double t[16];
#pragma unroll
        for (int c = 0; c < 16; ++c) t[c] = s_L[J][c0 + c];
#pragma unroll
        for (int c = 0; c < 16; ++c)
          if (c0 + c > J) r[c0 + c] -= l * t[c];
#pragma unroll
        for (int c = 0; c < 16; c += 8)
          asm volatile("" : "+v"(r[c0 + c]), "+v"(r[c0 + c + 1]), "+v"(r[c0 + c + 2]), "+v"(r[c0 + c + 3]),
                            "+v"(r[c0 + c + 4]), "+v"(r[c0 + c + 5]), "+v"(r[c0 + c + 6]), "+v"(r[c0 + c + 7]));
      }
    }
    chol_cols<J + 1>(lane, r, s_L, s_i, bad);
  }
}

// The diagonal block of step k of matrix blockIdx.x: its Cholesky factor's inverse to dinv[z][64][64]
__global__ __launch_bounds__(64) void k_chol_diag(int k, int ld, const double* __restrict__ A,
                                                  double* __restrict__ dinv, int* __restrict__ flag) {
  __shared__ double s_L[kNB][kNB + 2];
  __shared__ double s_i[kNB];
  if (*flag) return;
  const int z = blockIdx.x, lane = threadIdx.x;
  const double* a = A + mat_off(z, ld) + ((int64_t)k * kNB + lane) * ld + k * kNB;
  double r[kNB];
#pragma unroll
  for (int c = 0; c < kNB; c += 4) {
    const f64x4 v = *reinterpret_cast<const f64x4*>(a + c);
#pragma unroll
    for (int e = 0; e < 4; ++e) r[c + e] = v[e];
  }
  bool bad = false;
  chol_cols<0>(lane, r, s_L, s_i, bad);
  if (bad) {
    if (lane == 0) atomicOr(flag, 1);
    return;
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  // column `lane` of the inverse, forward substitution down the rows
#pragma unroll
  for (int i = 0; i < kNB; ++i) {
    double s0 = lane == i ? 1.0 : 0.0, s1 = 0.0;
#pragma unroll
    for (int t = 0; t < i; ++t) {
      if (t & 1) s1 -= s_L[t][i] * r[t];
      else s0 -= s_L[t][i] * r[t];
    }
    r[i] = (s0 + s1) * s_i[i];
    asm volatile("" ::: "memory");
  }
  double* out = dinv + (int64_t)z * kNB * kNB;
#pragma unroll
  for (int i = 0; i < kNB; ++i) out[i * kNB + lane] = r[i];
}

// Row blocks below the step's diagonal, and the identity's row blocks 0 .. k, times dinv^T, in place
__global__ __launch_bounds__(256) void k_chol_panel(int k, int nb, int ld, double* __restrict__ A,
                                                    const double* __restrict__ dinv, const int* __restrict__ flag) {
  if (*flag) return;
  const int below = nb - 1 - k;
  int b = blockIdx.x, z = 0;
  int64_t row;
  if (b < k + 1) {
    row = (int64_t)ld + (int64_t)b * kNB;   // the identity follows V
  } else {
    b -= k + 1;
    z = b / below;
    row = mat_off(z, ld) / ld + (int64_t)(k + 1 + b % below) * kNB;
  }
  const int wave = threadIdx.x >> 6, wr = 32 * (wave >> 1), wc = 32 * (wave & 1);
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  double* a = A + (row + wr) * ld + k * kNB;
  f64x4 acc[2][2] = {};
  nt_32x32(a, dinv + (int64_t)z * kNB * kNB + wc * kNB, ld, kNB, acc);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) a[(int64_t)(16 * i + lk + 4 * r) * ld + wc + 16 * j + li] = acc[i][j][r];
}

// Column blocks c > k: rows >= c of the three matrices and the identity's row blocks 0 .. k
__global__ __launch_bounds__(256) void k_chol_update(int k, int nb, int ld, double* __restrict__ A,
                                                     const int* __restrict__ flag) {
  if (*flag) return;
  const int c = k + 1 + blockIdx.y, z = blockIdx.z;   // z = 3: the identity
  const int b = blockIdx.x;
  int64_t row;
  if (z == 3) {
    if (b > k) return;
    row = (int64_t)ld + (int64_t)b * kNB;
  } else {
    if (c + b >= nb) return;
    row = mat_off(z, ld) / ld + (int64_t)(c + b) * kNB;
  }
  const int wave = threadIdx.x >> 6, wr = 32 * (wave >> 1), wc = 32 * (wave & 1);
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const double* crow = A + (mat_off(z == 3 ? 0 : z, ld) / ld + (int64_t)c * kNB + wc) * ld + k * kNB;
  double* a = A + (row + wr) * ld;
  f64x4 acc[2][2] = {};
  nt_32x32(a + k * kNB, crow, ld, ld, acc);
  double* o = a + (int64_t)c * kNB + wc;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) o[(int64_t)(16 * i + lk + 4 * r) * ld + 16 * j + li] -= acc[i][j][r];
}

// out[r][c] = in[r][c] (rows of ldi), or out[c][r] with tr, zero where in has no row or column
__global__ __launch_bounds__(256) void k_copy_pad(int nr, int nc, int64_t ldi, const double* __restrict__ in, int orows,
                                                  int64_t ldo, int tr, double* __restrict__ out) {
  __shared__ double s_t[32][33];
  const int x = threadIdx.x & 31, y = threadIdx.x >> 5;
  const int r0 = blockIdx.y * 32, c0 = blockIdx.x * 32;
  for (int i = y; i < 32; i += 8) {
    const bool in_ok = r0 + i < nr && c0 + x < nc;
    const double v = in[(int64_t)min(r0 + i, nr - 1) * ldi + min(c0 + x, nc - 1)];
    s_t[i][x] = in_ok ? v : 0.0;
  }
  __syncthreads();
  for (int i = y; i < 32; i += 8) {
    const int orow = tr ? c0 + i : r0 + i, ocol = tr ? r0 + x : c0 + x;
    if (orow < orows && ocol < ldo) out[(int64_t)orow * ldo + ocol] = tr ? s_t[x][i] : s_t[i][x];
  }
}

// B[(m, n)][q] = sum_P I3[(m, n)][P] W[q][P] over the pairs m >= n, to both orders of the pair. 128 pairs x 128
// q a workgroup, 64 x 64 a wavefront: both operands have k along their rows, so a wavefront's fragments of 8 k
// are 64-byte runs of its rows, loaded from global memory into registers while the 8 k before them multiply.
// L1 and L2 hold what the wavefronts share; LDS would add a copy and a barrier. Two wavefronts a SIMD: with one
// and three groups in flight the compiler moves the sums between both register files every turn (54 TF/s).
// tri: W is lower triangular (q, P), and a tile stops at its last q. Workgroup x runs on XCD x % 8: an XCD
// takes whole strips of pairs, their q tiles longest first, so a strip's integrals are read from HBM once. W:
// rows of ldw = 16 ceil(naux / 16), zero past naux and past nfit up to a whole tile.
// Bound by the matrix cores (63 TF/s): 18.4 ms for 480 functions and 2255 fitting functions, eigenvectors, where
// the product over both orders of a pair takes 33.3 ms at 70 TF/s; (H2O)_24 def2-TZVP, tri, 68 ms against 228.
__global__ __launch_bounds__(256, 2) void k_fit(int nao, int naux, int nfit, int64_t npair,
                                                const double* __restrict__ I3, const double* __restrict__ W, int ldw,
                                                int tri, double* __restrict__ B) {
  constexpr int MI = 4, TR = 32 * MI;   // tiles of 16 pairs a wavefront, pairs a workgroup
  __shared__ int64_t s_mn[TR], s_nm[TR];
  const int nqt = (nfit + 127) / 128;
  const int64_t ip = blockIdx.x / 8, strip = ip / nqt * 8 + blockIdx.x % 8, r0 = TR * strip;
  if (r0 >= npair) return;
  const int q0 = 128 * (nqt - 1 - (int)(ip % nqt));
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // uniform: no divergent loop around the sums
  const int wm = 16 * MI * (wave >> 1), wn = 64 * (wave & 1);
  if (tid < TR) {
    const int64_t r = min(r0 + tid, npair - 1);
    int64_t m = (int64_t)((sqrt(8.0 * (double)r + 1.0) - 1.0) * 0.5);
    while (m * (m + 1) / 2 > r) --m;
    while ((m + 1) * (m + 2) / 2 <= r) ++m;
    const int64_t n = r - m * (m + 1) / 2;
    s_mn[tid] = m * nao + n;
    s_nm[tid] = n * nao + m;
  }
  __syncthreads();
  const double* xa[MI];
#pragma unroll
  for (int i = 0; i < MI; ++i) xa[i] = I3 + s_mn[wm + 16 * i + li] * naux + 2 * lk;
  // W's rows by a uniform base and one 32-bit offset a lane: with the sums and two groups in flight the
  // registers are full
  const double* wrow = W + (int64_t)(q0 + wn) * ldw;
  const uint32_t woff = (uint32_t)(li * ldw + 2 * lk);
  const int kend = tri ? min(naux, q0 + wn + 64) : naux;
  const int ng = kend / 8, tail = kend % 8;   // tail: the last row's integrals end there
  f64x4 acc[MI][4] = {};
  f64x2u x[2][MI], y[2][4];
  const auto mul = [&](const f64x2u (&x)[MI], const f64x2u (&y)[4]) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[i][s], y[j][s], acc[i][j], 0, 0, 0);
  };
  const auto load = [&](int q, f64x2u (&x)[MI], f64x2u (&y)[4]) {   // group q from xa, wrow
#pragma unroll
    for (int i = 0; i < MI; ++i) x[i] = *reinterpret_cast<const f64x2u*>(xa[i] + 8 * q);
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] = *reinterpret_cast<const f64x2u*>(wrow + 16 * i * (int64_t)ldw + 8 * q + woff);
  };
  const auto step = [&](int n) {
#pragma unroll
    for (int i = 0; i < MI; ++i) xa[i] += 8 * n;
    wrow += 8 * n;
  };
  if (ng > 0) load(0, x[0], y[0]);
  int left = ng;
  for (; left >= 3; left -= 2) {
    load(1, x[1], y[1]);
    mul(x[0], y[0]);
    load(2, x[0], y[0]);
    mul(x[1], y[1]);
    step(2);
  }
  if (left > 1) load(1, x[1], y[1]);
  if (left > 0) mul(x[0], y[0]);
  if (left > 1) mul(x[1], y[1]);
  if (tail > 0) {
    step(left);
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const bool in = 2 * lk + s < tail;
        const double v = xa[i][in ? s : -2 * lk];   // clamped to the group's first
        x[0][i][s] = in ? v : 0.0;
      }
#pragma unroll
    for (int i = 0; i < 4; ++i) y[0][i] = *reinterpret_cast<const f64x2u*>(wrow + 16 * i * (int64_t)ldw + woff);
    mul(x[0], y[0]);
  }
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = wm + 16 * i + lk + 4 * r;
      if (r0 + row >= npair) continue;
      double *o1 = B + s_mn[row] * nfit, *o2 = B + s_nm[row] * nfit;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int q = q0 + wn + 16 * j + li;
        if (q < nfit) {
          o1[q] = acc[i][j][r];
          o2[q] = acc[i][j][r];
        }
      }
    }
}

}  // namespace

int metric_ld(int n) { return (n + kNB - 1) / kNB * kNB; }

// Words of launch_metric_chol's work array
size_t metric_chol_words(int n) { return 4 * (size_t)metric_ld(n) * metric_ld(n) + 3 * kNB * kNB; }

// C^-T of V = C C^T to Lt[P][q] (n x n) if every eigenvalue of V lies in (cutoff top, top); flag: 0 if so
hipError_t launch_metric_chol(int n, const double* V, double cutoff, double top, double* work, double* Lt, int* flag,
                              hipStream_t st) {
  const int ld = metric_ld(n), nb = ld / kNB;
  const int64_t nn = (int64_t)ld * ld;
  double* dinv = work + 4 * nn;
  hipLaunchKernelGGL(k_chol_start, dim3((unsigned)((nn + 255) / 256)), dim3(256), 0, st, n, ld, V, cutoff, top, work,
                     flag);
  for (int k = 0; k < nb; ++k) {
    hipLaunchKernelGGL(k_chol_diag, dim3(3), dim3(64), 0, st, k, ld, work, dinv, flag);
    const int below = nb - 1 - k;
    hipLaunchKernelGGL(k_chol_panel, dim3((unsigned)(k + 1 + 3 * below)), dim3(256), 0, st, k, nb, ld, work, dinv,
                       flag);
    if (below > 0)
      hipLaunchKernelGGL(k_chol_update, dim3((unsigned)std::max(k + 1, below), (unsigned)below, 4), dim3(256), 0, st, k,
                         nb, ld, work, flag);
  }
  const unsigned t = (unsigned)((n + 31) / 32);
  hipLaunchKernelGGL(k_copy_pad, dim3(t, t), dim3(256), 0, st, n, n, (int64_t)ld, work + nn, n, (int64_t)n, 0, Lt);
  return hipGetLastError();
}

// Words of launch_fit's copy of the factor
size_t fit_words(int naux, int nfit) { return (size_t)((nfit + 127) / 128 * 128) * ((naux + 15) / 16 * 16); }

// B[mn][q] = sum_P I3[mn][P] Lt[P][q] (rows of nfit); tri: Lt[P][q] = 0 for P > q
hipError_t launch_fit(int nao, int naux, int nfit, const double* I3, const double* Lt, int tri, double* W, double* B,
                      hipStream_t st) {
  if (nao == 0 || nfit == 0) return hipSuccess;
  const int ldw = (naux + 15) / 16 * 16, nqt = (nfit + 127) / 128;
  hipLaunchKernelGGL(k_copy_pad, dim3((unsigned)(nqt * 4), (unsigned)((ldw + 31) / 32)), dim3(256), 0, st, naux, nfit,
                     (int64_t)nfit, Lt, nqt * 128, (int64_t)ldw, 1, W);
  const int64_t npair = (int64_t)nao * (nao + 1) / 2;
  const int64_t strips = (npair + 127) / 128;
  hipLaunchKernelGGL(k_fit, dim3((unsigned)((strips + 7) / 8 * 8 * nqt)), dim3(256), 0, st, nao, naux, nfit, npair, I3,
                     W, ldw, tri, B);
  return hipGetLastError();
}

}  // namespace dfks
