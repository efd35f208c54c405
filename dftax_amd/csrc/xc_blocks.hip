// FP64 products of the XC term on the compact grid, all blocks in one launch.
//
// Block b holds 128 grid points and the n functions cols[0..n) that reach them
// (n a multiple of 32, -1 pads past the first nf); its AO planes are ao[k plane + g n + i].
//   k_xcb_rho  Z = Phi P_b over a strip of at most 64 columns, reduced at once to the
//              strip's share of rho and grad rho, so Z is never stored
//   k_xcb_v    Vh_b = Phi^T W over a strip, W = a phi + b . grad phi formed in LDS
// (the pointwise functional between them is k_xcb_point* in xc.hip). One
// workgroup takes one strip; workgroup x runs on XCD x % 8, and the strips of a
// block are 8 ids apart, so they share that XCD's L2 for the block's AO rows and
// the blocks of every width spread over the XCDs. Blocks come widest first.
//
// (H2O)_24 def2-TZVP on the MI355X: rho 4.0 ms, the pointwise pass 0.2 ms, Vh
// 3.85 ms, against 14 ms for the per-bin gathers, batched products and
// wavefront-per-point kernels they replace. Vh is near what its AO rows read
// and products written take at the copy rate (3 ms); rho is between its reads
// (1.7 ms) and its matrix work (2.8 ms). An MFMA sums over any order of k as
// long as both operands agree, so the operand that is contiguous along k (Phi
// in Z) is loaded straight from global memory in 32-byte runs, lane group l
// taking k = 4 l + s in step s, and the other operand sits in LDS in fragment
// order (64 consecutive doubles per step and 16 columns): no conflicts and no
// transposition. In Vh the contraction runs over the points, so Phi's
// fragments are 128-byte runs of one point's row as they lie.
#include <cstdint>

#include "dfks_common.h"

namespace dfks {

namespace {

typedef double dbl2 __attribute__((ext_vector_type(2)));
typedef double dbl4 __attribute__((ext_vector_type(4)));

constexpr int kG = 128;      // points per block
constexpr int kKC = 32;      // functions of P staged per step

// sum over the 16 lanes of a row, in every lane of it
template <int CTRL>
__device__ __forceinline__ double dpp_add(double x) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, false);
  return x + __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double row_sum(double x) {
  x = dpp_add<0x128>(x);   // rotate right by 8, 4, 2, 1 within the row
  x = dpp_add<0x124>(x);
  x = dpp_add<0x122>(x);
  return dpp_add<0x121>(x);
}

// One strip of NJ 16-column groups of Z. Wavefront w owns points 32 w .. 32 w + 31.
template <int NJ>
__device__ __forceinline__ void rho_strip(const XcBlock& b, int c0, const double* __restrict__ ao,
                                          const int32_t* __restrict__ cols, const double* __restrict__ P, int64_t nao,
                                          double* __restrict__ part, double* __restrict__ s_p) {
  constexpr int W = 16 * NJ, PER = kKC * W / 256, STEP = 256 / W;   // P values a thread stages, k apart
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = b.n;
  const int pc = tid % W, pk = tid / W;
  const int32_t cc = cols[c0 + pc];
  const double* pcol = P + max(cc, 0);
  const double* arow = ao + (int64_t)(32 * wv + li) * n + 4 * lk;
  dbl4 acc[2][NJ];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = dbl4{0.0, 0.0, 0.0, 0.0};
  double p[PER];
  dbl2 a[2][2][2];   // k half, point group, pair of k
  const auto load_p = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < PER; ++e) p[e] = pcol[(int64_t)max(cols[k0 + pk + STEP * e], 0) * nao];
  };
  const auto load_a = [&](int q, int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const dbl2* src = reinterpret_cast<const dbl2*>(arow + (int64_t)16 * i * n + k0 + 16 * q);
      a[q][i][0] = src[0];
      a[q][i][1] = src[1];
    }
  };
  load_p(0);
  load_a(0, 0);
  load_a(1, 0);
  for (int k0 = 0, buf = 0; k0 < n; k0 += kKC, buf ^= 1) {
    double* sp = s_p + buf * (kKC * 64);
    if (k0 + kKC > b.nf || c0 + W > b.nf) {   // padded k and columns: zero, whatever P[0][.] and P[.][0] hold
#pragma unroll
      for (int e = 0; e < PER; ++e)
        if (k0 + pk + STEP * e >= b.nf || c0 + pc >= b.nf) p[e] = 0.0;
    }
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int k = pk + STEP * e;   // its step (k / 16, k % 4) and lane group (k % 16) / 4
      sp[(((k >> 4) * 4 + (k & 3)) * NJ + pc % NJ) * 64 + ((k >> 2) & 3) * 16 + pc / NJ] = p[e];
    }
    __syncthreads();   // the other buffer's readers passed the previous barrier
    const bool more = k0 + kKC < n;
    if (more) load_p(k0 + kKC);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        double bf[NJ];
#pragma unroll
        for (int j = 0; j < NJ; ++j) bf[j] = sp[((q * 4 + s) * NJ + j) * 64 + lane];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < NJ; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[q][i][s >> 1][s & 1], bf[j], acc[i][j], 0, 0, 0);
      }
      if (more) load_a(q, k0 + kKC);
    }
  }
  // result register r: point 32 w + 16 i + lk + 4 r, column c0 + NJ li + j (the lane's own NJ columns in a row)
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int g = 32 * wv + 16 * i + lk + 4 * r;
      const double* src = ao + (int64_t)g * n + c0 + NJ * li;
      double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int j = 0; j < NJ; j += 2) {
          const dbl2 x = *reinterpret_cast<const dbl2*>(src + k * b.plane + j);
          s[k] += acc[i][j][r] * x[0] + acc[i][j + 1][r] * x[1];
        }
#pragma unroll
      for (int k = 0; k < 4; ++k) s[k] = row_sum(s[k]);
      const double o = li == 0 ? s[0] : (li == 1 ? s[1] : (li == 2 ? s[2] : s[3]));
      if (li < 4) part[li * kG + g] = o;
    }
}

__global__ __launch_bounds__(256, 3) void k_xcb_rho(const XcBlock* __restrict__ blks, const int32_t* __restrict__ wgs,
                                                 const double* __restrict__ ao, const int32_t* __restrict__ cols,
                                                 const double* __restrict__ P, int64_t nao,
                                                 double* __restrict__ part) {
  __shared__ double s_p[2 * kKC * 64];
  const int32_t id = wgs[blockIdx.x];
  if (id < 0) return;
  const int strip = id & (kXcbStrips - 1);
  const XcBlock b = blks[id / kXcbStrips];
  const int c0 = 64 * strip;
  double* dst = part + (b.part0 + strip) * (4 * kG);
  if (b.n - c0 >= 64) rho_strip<4>(b, c0, ao + b.ao0, cols + b.col0, P, nao, dst, s_p);
  else rho_strip<2>(b, c0, ao + b.ao0, cols + b.col0, P, nao, dst, s_p);
}

// One strip of NJ 16-column groups of Vh_b: wavefront w takes the 32-row groups w, w + 4, ...
template <int NJ>
__device__ __forceinline__ void v_strip(const XcBlock& b, int c0, const double* __restrict__ ao,
                                        const double* __restrict__ coef, double* __restrict__ q,
                                        double* __restrict__ s_w) {
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = b.n;
  // W: thread t takes two columns of the points t / (8 NJ), ...
  constexpr int CP = 8 * NJ, GS = 256 / CP;
  const int cg = 2 * (tid % CP);
#pragma unroll 4
  for (int g = tid / CP; g < kG; g += GS) {
    const double* src = ao + (int64_t)g * n + c0 + cg;
    const dbl4 cf = *reinterpret_cast<const dbl4*>(coef + 4 * g);
    const dbl2 x0 = *reinterpret_cast<const dbl2*>(src), x1 = *reinterpret_cast<const dbl2*>(src + b.plane),
               x2 = *reinterpret_cast<const dbl2*>(src + 2 * b.plane),
               x3 = *reinterpret_cast<const dbl2*>(src + 3 * b.plane);
    dbl2 w;
#pragma unroll
    for (int e = 0; e < 2; ++e) w[e] = cf[0] * x0[e] + cf[1] * x1[e] + cf[2] * x2[e] + cf[3] * x3[e];
    *reinterpret_cast<dbl2*>(s_w + ((g >> 2) * NJ + (cg >> 4)) * 64 + (g & 3) * 16 + (cg & 15)) = w;
  }
  __syncthreads();
  for (int m0 = 32 * wv; m0 < n; m0 += 128) {
    dbl4 acc[2][NJ];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] = dbl4{0.0, 0.0, 0.0, 0.0};
    const double* arow = ao + (int64_t)lk * n + m0 + 2 * li;   // step s: point 4 s + lk, functions 2 li + i
    const int64_t ds = (int64_t)4 * n;
    constexpr int D = 4;               // steps of Phi in flight
    dbl2 a[D];
#pragma unroll
    for (int d = 0; d < D; ++d) a[d] = *reinterpret_cast<const dbl2*>(arow + d * ds);
#pragma unroll 1
    for (int s0 = 0; s0 < kG / 4; s0 += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        const int s = s0 + d;
        double bf[NJ];
#pragma unroll
        for (int j = 0; j < NJ; ++j) bf[j] = s_w[(s * NJ + j) * 64 + lane];
        const double f0 = a[d][0], f1 = a[d][1];
        const int sn = s + D < kG / 4 ? s + D : s;       // past the end: reload, unused
        a[d] = *reinterpret_cast<const dbl2*>(arow + sn * ds);
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[0][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(f0, bf[j], acc[0][j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[1][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(f1, bf[j], acc[1][j], 0, 0, 0);
      }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        // result register r: function 2 (lk + 4 r) + i of the group, columns c0 + 16 j + li
        double* dst = q + (int64_t)(m0 + 2 * (lk + 4 * r) + i) * n + c0 + li;
#pragma unroll
        for (int j = 0; j < NJ; ++j) dst[16 * j] = acc[i][j][r];
      }
  }
}

__global__ __launch_bounds__(256, 2) void k_xcb_v(const XcBlock* __restrict__ blks, const int32_t* __restrict__ wgs,
                                               const double* __restrict__ ao, const double* __restrict__ coef,
                                               double* __restrict__ q) {
  __shared__ __attribute__((aligned(16))) double s_w[kG * 64];
  const int32_t id = wgs[blockIdx.x];
  if (id < 0) return;
  const int strip = id & (kXcbStrips - 1);
  const XcBlock b = blks[id / kXcbStrips];
  const int c0 = 64 * strip;
  const double* cf = coef + 4 * b.pt0;
  if (b.n - c0 >= 64) v_strip<4>(b, c0, ao + b.ao0, cf, q + b.q0, s_w);
  else v_strip<2>(b, c0, ao + b.ao0, cf, q + b.q0, s_w);
}

}  // namespace

// part[(part0 + strip)][4][128]: the strip's share of sum_c Z phi, Z d_x phi, d_y, d_z per point
hipError_t launch_xcb_rho(const XcBlock* blks, const int32_t* wgs, int nwg, const double* ao, const int32_t* cols,
                          const double* P, int64_t nao, double* part, hipStream_t st) {
  if (nwg == 0) return hipSuccess;
  if ((uintptr_t)ao % 16 != 0) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_xcb_rho, dim3((unsigned)nwg), dim3(256), 0, st, blks, wgs, ao, cols, P, nao, part);
  return hipGetLastError();
}

// coef[4 point ..] = {a, bx, by, bz} of W, q the block products
hipError_t launch_xcb_v(const XcBlock* blks, const int32_t* wgs, int nwg, const double* ao, const double* coef,
                        double* q, hipStream_t st) {
  if (nwg == 0) return hipSuccess;
  if ((uintptr_t)ao % 16 != 0 || (uintptr_t)coef % 32 != 0) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_xcb_v, dim3((unsigned)nwg), dim3(256), 0, st, blks, wgs, ao, coef, q);
  return hipGetLastError();
}

}  // namespace dfks
