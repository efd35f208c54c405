// The plan of the compact XC grid, on the device: points in Morton order, blocks of kXcG of them, the
// shells that reach each block, and from these the blocks' columns and the row lists of the Vxc assembly.
//
// The same lists as a host program that walks points, blocks and shells in order: keys and distances are
// formed with the same FP64 operations (no contraction), sums run in the order of the points, the sort is
// stable, and every list position is a count of what comes before. Bound by launches and the copies of the
// points. Sort, scans and lists of (H2O)_8 def2-TZVP 1.4 ms (9.1 on the host with 4 threads), of a tree of 20
// heavy atoms 2.7 ms (35), of (H2O)_24 3.8 ms (52).
// Reference: dftax/ks/grid blocks (dftax/energy/xc.py), whose grid is one dense array.
#include <algorithm>
#include <cstdint>

#include "dfks_common.h"

namespace dfks {

namespace {

constexpr int kTile = 2048;   // points a wavefront sorts: ten ballots for 64 of them, one atomic-free pass
constexpr int kDigits = 1024;
constexpr int kBoundBlocks = 256;

__device__ __forceinline__ void wave_fence() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }

// part[block] = {lo x y z, hi x y z} of the block's share of the points
__global__ __launch_bounds__(256) void k_plan_bounds(int64_t ng, const double* __restrict__ X,
                                                     double* __restrict__ part) {
  __shared__ double s[6][256];
  double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
  for (int64_t g = blockIdx.x * (int64_t)256 + threadIdx.x; g < ng; g += (int64_t)gridDim.x * 256)
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double x = X[3 * g + d];
      lo[d] = x < lo[d] ? x : lo[d];
      hi[d] = x > hi[d] ? x : hi[d];
    }
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    s[d][threadIdx.x] = lo[d];
    s[3 + d][threadIdx.x] = hi[d];
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    const bool up = threadIdx.x >= 3;
    double v = s[threadIdx.x][0];
    for (int i = 1; i < 256; ++i) {
      const double x = s[threadIdx.x][i];
      if (up ? x > v : x < v) v = x;
    }
    part[blockIdx.x * 6 + threadIdx.x] = v;
  }
}

__device__ __forceinline__ uint32_t spread3(uint32_t x) {
  x &= 0x3ff;
  x = (x | (x << 16)) & 0x030000ff;
  x = (x | (x << 8)) & 0x0300f00f;
  x = (x | (x << 4)) & 0x030c30c3;
  x = (x | (x << 2)) & 0x09249249;
  return x;
}

__global__ __launch_bounds__(256) void k_plan_keys(int64_t ng, const double* __restrict__ X, int nparts,
                                                   const double* __restrict__ part, uint32_t* __restrict__ key,
                                                   int32_t* __restrict__ idx) {
#pragma clang fp contract(off)
  __shared__ double s[6];
  if (threadIdx.x < 6) {
    const bool up = threadIdx.x >= 3;
    double v = part[threadIdx.x];
    for (int i = 1; i < nparts; ++i) {
      const double x = part[i * 6 + threadIdx.x];
      if (up ? x > v : x < v) v = x;
    }
    s[threadIdx.x] = v;
  }
  __syncthreads();
  const int64_t g = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (g >= ng) return;
  uint32_t c = 0;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const double t = (X[3 * g + d] - s[d]) / (s[3 + d] - s[d] + 1e-12), u = t * 1023.0;
    const double v = u > 0.0 ? u : 0.0;
    c |= spread3((uint32_t)(v < 1023.0 ? v : 1023.0)) << d;
  }
  key[g] = c;
  idx[g] = (int32_t)g;
}

// cnt[digit][tile], one wavefront a tile
__global__ __launch_bounds__(64) void k_radix_count(int64_t ng, int shift, const uint32_t* __restrict__ key, int ntile,
                                                    int32_t* __restrict__ cnt) {
  __shared__ int32_t s[kDigits];
  for (int i = threadIdx.x; i < kDigits; i += 64) s[i] = 0;
  __syncthreads();
  const int64_t g0 = (int64_t)blockIdx.x * kTile, g1 = min(ng, g0 + kTile);
  for (int64_t g = g0 + threadIdx.x; g < g1; g += 64) atomicAdd(&s[(key[g] >> shift) & (kDigits - 1)], 1);
  __syncthreads();
  for (int i = threadIdx.x; i < kDigits; i += 64) cnt[(int64_t)i * ntile + blockIdx.x] = s[i];
}

// cnt[digit][.] to its exclusive sums over the tiles, the total to tot; one wavefront a digit
__global__ __launch_bounds__(64) void k_radix_scan(int ntile, int32_t* __restrict__ cnt, int32_t* __restrict__ tot) {
  int32_t* c = cnt + (int64_t)blockIdx.x * ntile;
  int32_t run = 0;
  for (int t0 = 0; t0 < ntile; t0 += 64) {
    const int t = t0 + threadIdx.x;
    const int32_t v = t < ntile ? c[t] : 0;
    int32_t x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int32_t y = __shfl_up(x, o);
      if ((int)threadIdx.x >= o) x += y;
    }
    if (t < ntile) c[t] = run + x - v;
    run += __shfl(x, 63);
  }
  if (threadIdx.x == 0) tot[blockIdx.x] = run;
}

// A tile's points to their places, 64 at a time in order: a lane's place is its digit's next one plus the number of
// earlier lanes with the same digit
__global__ __launch_bounds__(64) void k_radix_scatter(int64_t ng, int shift, const uint32_t* __restrict__ kin,
                                                      const int32_t* __restrict__ vin, int ntile,
                                                      const int32_t* __restrict__ cnt, const int32_t* __restrict__ tot,
                                                      uint32_t* __restrict__ kout, int32_t* __restrict__ vout) {
  __shared__ int32_t s[kDigits];
  const int lane = threadIdx.x;
  int32_t run = 0;
  for (int d0 = 0; d0 < kDigits; d0 += 64) {   // digits before this one, and this digit in the tiles before
    const int32_t v = tot[d0 + lane];
    int32_t x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int32_t y = __shfl_up(x, o);
      if (lane >= o) x += y;
    }
    s[d0 + lane] = run + x - v + cnt[(int64_t)(d0 + lane) * ntile + blockIdx.x];
    run += __shfl(x, 63);
  }
  wave_fence();
  const int64_t g0 = (int64_t)blockIdx.x * kTile;
  for (int k = 0; k < kTile && g0 + k < ng; k += 64) {
    const int64_t g = g0 + k + lane;
    const bool in = g < ng;
    const uint32_t key = in ? kin[g] : 0u;
    const int32_t val = in ? vin[g] : 0;
    const uint32_t d = (key >> shift) & (kDigits - 1);
    uint64_t same = __ballot(in);
#pragma unroll
    for (int b = 0; b < 10; ++b) {
      const uint64_t m = __ballot((d >> b) & 1u);
      same &= (d >> b) & 1u ? m : ~m;
    }
    const int before = __popcll(same & ((1ull << lane) - 1ull));
    const int32_t at = s[d] + before;
    wave_fence();
    if (in && before == 0) s[d] = at + __popcll(same);
    wave_fence();
    if (in) {
      kout[at] = key;
      vout[at] = val;
    }
  }
}

// A block's shells, one wavefront a block: first column of each shell that reaches it, -1 else (loc[block][shell]),
// its numbers of functions and of shells, and each shell's number of blocks
__global__ __launch_bounds__(64) void k_plan_scan(int64_t ng, const double* __restrict__ X,
                                                  const int32_t* __restrict__ idx, ShellSet S,
                                                  const double* __restrict__ rcut, int32_t* __restrict__ loc,
                                                  int32_t* __restrict__ nfn, int32_t* __restrict__ nshell,
                                                  int32_t* __restrict__ nblk_of) {
#pragma clang fp contract(off)
  __shared__ double s_x[kXcG][3];
  __shared__ double s_c[3];
  const int lane = threadIdx.x;
  const int64_t b = blockIdx.x, p0 = b * kXcG, p1 = min(ng, p0 + kXcG);
  const int np = (int)(p1 - p0);
  for (int i = lane; i < 3 * np; i += 64) s_x[i / 3][i % 3] = X[3 * (int64_t)idx[p0 + i / 3] + i % 3];
  __syncthreads();
  if (lane < 3) {
    double c = 0.0;
    for (int p = 0; p < np; ++p) c += s_x[p][lane];
    s_c[lane] = c / (double)np;
  }
  __syncthreads();
  const double c0 = s_c[0], c1 = s_c[1], c2 = s_c[2];
  double rad = 0.0;
  for (int p = lane; p < np; p += 64) {
    const double x = s_x[p][0] - c0, y = s_x[p][1] - c1, z = s_x[p][2] - c2, r = sqrt(x * x + y * y + z * z);
    rad = r > rad ? r : rad;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const double r = __shfl_xor(rad, o);
    rad = r > rad ? r : rad;
  }
  int col = 0, ns = 0;
  for (int s0 = 0; s0 < S.n; s0 += 64) {
    const int s = s0 + lane;
    bool hit = false;
    int nf = 0;
    if (s < S.n && rcut[s] >= 0.0) {
      const double x = S.centre[3 * s] - c0, y = S.centre[3 * s + 1] - c1, z = S.centre[3 * s + 2] - c2;
      hit = sqrt(x * x + y * y + z * z) - rad <= rcut[s];
      nf = hit ? nfun(S.l[s], S.spherical) : 0;
    }
    int at = nf;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(at, o);
      if (lane >= o) at += y;
    }
    if (s < S.n) loc[b * S.n + s] = hit ? col + at - nf : -1;
    if (hit) atomicAdd(&nblk_of[s], 1);
    col += __shfl(at, 63);
    ns += __popcll(__ballot(hit));
  }
  if (lane == 0) {
    nfn[b] = col;
    nshell[b] = ns;
  }
}

// Block ob of the plan (Morton block order[ob], width w[ob], columns from col0[ob]): points and weights (a short
// block repeats its last point with weight 0), columns (-1 past the block's functions) and shell list
__global__ __launch_bounds__(64) void k_plan_fill(int64_t ng, const double* __restrict__ X,
                                                  const double* __restrict__ gw, const int32_t* __restrict__ idx,
                                                  ShellSet S, const int32_t* __restrict__ loc,
                                                  const int32_t* __restrict__ order,
                                                  const int32_t* __restrict__ w, const int64_t* __restrict__ col0,
                                                  const int64_t* __restrict__ shoff, double* __restrict__ pts,
                                                  double* __restrict__ wts, int32_t* __restrict__ cols,
                                                  int2* __restrict__ shl) {
  const int lane = threadIdx.x;
  const int64_t ob = blockIdx.x, b = order[ob], p0 = b * kXcG, p1 = min(ng, p0 + kXcG);
  for (int i = lane; i < 3 * kXcG; i += 64)
    pts[3 * ob * kXcG + i] = X[3 * (int64_t)idx[min(p0 + i / 3, p1 - 1)] + i % 3];
  for (int p = lane; p < kXcG; p += 64) wts[ob * kXcG + p] = p0 + p < p1 ? gw[idx[p0 + p]] : 0.0;
  int32_t* cb = cols + col0[ob];
  int64_t at = shoff[ob];
  int end = 0;
  for (int s0 = 0; s0 < S.n; s0 += 64) {
    const int s = s0 + lane, c = s < S.n ? loc[b * S.n + s] : -1;
    const uint64_t hit = __ballot(c >= 0);
    int last = 0;
    if (c >= 0) {
      shl[at + __popcll(hit & ((1ull << lane) - 1ull))] = make_int2(s, c);
      const int nf = nfun(S.l[s], S.spherical);
      for (int f = 0; f < nf; ++f) cb[c + f] = S.ao0[s] + f;
      last = c + nf;
    }
    at += __popcll(hit);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) last = max(last, __shfl_xor(last, o));
    end = max(end, last);
  }
  for (int i = end + lane; i < w[ob]; i += 64) cb[i] = -1;
}

// Row lists of the Vxc assembly, one wavefront a shell: for its function f, the blocks it reaches in plan order from
// vrow[ao0 + f] (product row, first column, width)
__global__ __launch_bounds__(64) void k_plan_rows(int64_t nblk, ShellSet S, const int32_t* __restrict__ loc,
                                                  const int32_t* __restrict__ order, const int32_t* __restrict__ w,
                                                  const int64_t* __restrict__ col0, const int64_t* __restrict__ q0,
                                                  const int64_t* __restrict__ vrow, int64_t* __restrict__ vprow,
                                                  int64_t* __restrict__ vpcol, int32_t* __restrict__ vlen) {
  const int lane = threadIdx.x, s = blockIdx.x;
  const int nf = nfun(S.l[s], S.spherical);
  int64_t run = 0;
  for (int64_t o0 = 0; o0 < nblk; o0 += 64) {
    const int64_t ob = o0 + lane;
    const int c = ob < nblk ? loc[(int64_t)order[ob] * S.n + s] : -1;
    const uint64_t hit = __ballot(c >= 0);
    if (c >= 0) {
      const int64_t at = run + __popcll(hit & ((1ull << lane) - 1ull)), qb = q0[ob], cb = col0[ob];
      const int n = w[ob];
      for (int f = 0; f < nf; ++f) {
        const int64_t e = vrow[S.ao0[s] + f] + at;
        vprow[e] = qb + (int64_t)(c + f) * n;
        vpcol[e] = cb;
        vlen[e] = n;
      }
    }
    run += __popcll(hit);
  }
}

}  // namespace

// 4-byte words of launch_plan_sort's work space: two keys and two indices a point, the digits' counts
size_t plan_sort_words(int64_t ng) {
  return 4 * (size_t)ng + kDigits * (size_t)((ng + kTile - 1) / kTile + 1) + 12 * kBoundBlocks + 2;
}

// The points' indices in the order of their 30-bit Morton keys (equal keys in their own order); *idx points into work
hipError_t launch_plan_sort(int64_t ng, const double* X, uint32_t* work, const int32_t** idx, hipStream_t st) {
  const int ntile = (int)((ng + kTile - 1) / kTile);
  double* part = reinterpret_cast<double*>(work);   // the allocation starts on a double
  uint32_t* k[2] = {work + 12 * kBoundBlocks, work + 12 * kBoundBlocks + ng};
  int32_t* v[2] = {reinterpret_cast<int32_t*>(k[1] + ng), reinterpret_cast<int32_t*>(k[1] + 2 * ng)};
  int32_t *cnt = v[1] + ng, *tot = cnt + (int64_t)kDigits * ntile;
  const unsigned nb = (unsigned)((ng + 255) / 256);
  const int np = (int)std::min<unsigned>(kBoundBlocks, nb);
  hipLaunchKernelGGL(k_plan_bounds, dim3((unsigned)np), dim3(256), 0, st, ng, X, part);
  hipLaunchKernelGGL(k_plan_keys, dim3(nb), dim3(256), 0, st, ng, X, np, part, k[0], v[0]);
  for (int pass = 0; pass < 3; ++pass) {
    const int a = pass & 1, b = a ^ 1;
    hipLaunchKernelGGL(k_radix_count, dim3((unsigned)ntile), dim3(64), 0, st, ng, 10 * pass, k[a], ntile, cnt);
    hipLaunchKernelGGL(k_radix_scan, dim3(kDigits), dim3(64), 0, st, ntile, cnt, tot);
    hipLaunchKernelGGL(k_radix_scatter, dim3((unsigned)ntile), dim3(64), 0, st, ng, 10 * pass, k[a], v[a], ntile, cnt,
                       tot, k[b], v[b]);
  }
  *idx = v[1];
  return hipGetLastError();
}

hipError_t launch_plan_scan(int64_t ng, const double* X, const int32_t* idx, const ShellSet& S, const double* rcut,
                            int32_t* loc, int32_t* nfn, int32_t* nshell, int32_t* nblk_of, hipStream_t st) {
  hipLaunchKernelGGL(k_plan_scan, dim3((unsigned)((ng + kXcG - 1) / kXcG)), dim3(64), 0, st, ng, X, idx, S, rcut, loc,
                     nfn, nshell, nblk_of);
  return hipGetLastError();
}

hipError_t launch_plan_fill(int64_t ng, const double* X, const double* gw, const int32_t* idx, const ShellSet& S,
                            const int32_t* loc, const int32_t* order, const int32_t* w, const int64_t* col0,
                            const int64_t* shoff, double* pts, double* wts, int32_t* cols, int2* shl, hipStream_t st) {
  hipLaunchKernelGGL(k_plan_fill, dim3((unsigned)((ng + kXcG - 1) / kXcG)), dim3(64), 0, st, ng, X, gw, idx, S, loc,
                     order, w, col0, shoff, pts, wts, cols, shl);
  return hipGetLastError();
}

hipError_t launch_plan_rows(int64_t nblk, const ShellSet& S, const int32_t* loc, const int32_t* order, const int32_t* w,
                            const int64_t* col0, const int64_t* q0, const int64_t* vrow, int64_t* vprow, int64_t* vpcol,
                            int32_t* vlen, hipStream_t st) {
  hipLaunchKernelGGL(k_plan_rows, dim3((unsigned)S.n), dim3(64), 0, st, nblk, S, loc, order, w, col0, q0, vrow, vprow,
                     vpcol, vlen);
  return hipGetLastError();
}

}  // namespace dfks
