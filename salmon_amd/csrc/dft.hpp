// 3-D DFTs of one grid in three launches: a plane's z and y transforms, the x
// transforms forward, times a multiplier, and back, and a plane's y and z
// transforms back.  For the Hartree potential (scf.hpp) and the kinetic
// preconditioner (cg.hpp), whose grids are so small that an axis per launch, with
// its conversion and multiplier passes, was nine and five launches of 4 to 7 us of
// start, load latency and end each; a self-consistent step of 64 k x 32 bands of
// 16^3 took 250 us, 50 of them for these.
//
// Sums are direct (grid axes are any length, at most a few dozen points), with
// twiddles (cos, sin)(2 pi j / n) from a table.  A plane is shared by several
// blocks without repeating work: the first of its two transforms is formed only
// for the second axis' lines that the block transforms next.
#pragma once
#include <algorithm>

#include "common.hpp"

namespace salmon {
namespace dft {

constexpr int kTile = 1024;  // grid values staged at a time
constexpr int kLines = 8;    // lines of a block's second transform (256 threads; more on short axes)
constexpr int kBlocks = 512;

// Lines per block of a plane launch for axes of the given lengths: a value per
// thread, and up to kLines where that leaves two blocks per compute unit.  Few
// planes of long lines have too few blocks otherwise: eight planes of 8x256 took 183
// us for the whole solve with kLines, 101 so (a pass per axis 141); 256 and 1024 for
// kBlocks took 1.18 and 1.33 ms on ten planes of 200x200, 512 1.05.
inline int plane_lines(int first, int second, long planes) {
  int nl = std::max(1, 256 / second);
  while (nl < kLines && planes * ((first + nl) / (nl + 1)) >= kBlocks) ++nl;
  return nl;
}
// dynamic LDS of the plane kernels with nl lines
inline size_t plane_lds(int first, int second, int nl) {
  return 16 * ((size_t)std::max(kTile, first) + (size_t)nl * second + first + second);
}

// sum over m = m0, m0 + dm, ... of a(m) e^{sgn 2 pi i e m / n}, a(m) at a[m * as]
__device__ __forceinline__ cplx<double> line_sum(const cplx<double>* a, int as, int n, int e, const double2* w, double sgn,
                                                 int m0 = 0, int dm = 1) {
  double re = 0.0, im = 0.0;
  int j = m0 == 0 ? 0 : e * m0 % n;
  const int dj = dm == 1 ? e : e * dm % n;
#pragma unroll 4
  for (int m = m0; m < n; m += dm) {
    const double c = w[j].x, s = sgn * w[j].y;
    const cplx<double> v = a[m * as];
    re += c * v.re - s * v.im;
    im += c * v.im + s * v.re;
    j += dj;
    if (j >= n) j -= n;
  }
  return {re, im};
}

// Both transforms of a plane for nl lines of the second axis.  The
// plane's value at (first axis a, second axis b) comes from in(a, b), tiles of
// whole first-axis lines at a time; out(a, b, value) gets the results of the
// block's nl lines a = blockIdx.x * nl ...  FAST: the first axis is
// the one of consecutive grid points.
template <bool FAST, typename IN, typename OUT>
__device__ __forceinline__ void plane(int NA, int NB, int nl, const double* twa, const double* twb, double sgn, IN in, OUT out) {
  extern __shared__ __align__(16) unsigned char dft_lds[];
  cplx<double>* tile = (cplx<double>*)dft_lds;
  const int a0 = blockIdx.x * nl, na = min(nl, NA - a0), t = threadIdx.x;
  cplx<double>* mid = tile + max(kTile, NA);  // (b, a): first transform's results
  double2* wa = (double2*)(mid + nl * NB);
  double2* wb = wa + NA;
  for (int j = t; j < NA; j += 256) wa[j] = make_double2(twa[2 * j], twa[2 * j + 1]);
  for (int j = t; j < NB; j += 256) wb[j] = make_double2(twb[2 * j], twb[2 * j + 1]);
  const int rows = max(1, kTile / NA);  // first-axis lines per tile
  for (int b0 = 0; b0 < NB; b0 += rows) {
    const int nb = min(rows, NB - b0);
    __syncthreads();
    for (int i = t; i < nb * NA; i += 256) {
      const int a = FAST ? i % NA : i / nb, b = FAST ? i / NA : i % nb;
      tile[b * NA + a] = in(a, b0 + b);
    }
    __syncthreads();
    // long lines leave few sums a tile: neighbouring lanes share each (ten planes of
    // 200x200 1.47 -> 1.05 ms)
    int parts = 1;
    while (parts < 8 && 2 * parts * nb * na <= 256 && NA > 32 * parts) parts *= 2;
    if (parts == 1) {
      for (int i = t; i < nb * na; i += 256) {
        const int b = i / na, a = i - b * na;
        mid[(b0 + b) * na + a] = line_sum(tile + b * NA, 1, NA, a0 + a, wa, sgn);
      }
      continue;
    }
    for (int i = t; i < nb * na * parts; i += 256) {
      const int o = i / parts, b = o / na, a = o - b * na;
      cplx<double> v = line_sum(tile + b * NA, 1, NA, a0 + a, wa, sgn, i - o * parts, parts);
      for (int s = 1; s < parts; s *= 2) {
        v.re += __shfl_xor(v.re, s);
        v.im += __shfl_xor(v.im, s);
      }
      if (i == o * parts) mid[(b0 + b) * na + a] = v;
    }
  }
  __syncthreads();
  for (int i = t; i < NB * na; i += 256) {
    const int b = FAST ? i / na : i % NB, a = FAST ? i - b * na : i / NB;
    out(a0 + a, b, line_sum(mid + a, na, NB, b, wb, sgn));
  }
}

// The x lines of a grid: forward, times mul(x, y, z), back.  In place, 256 / NLx
// lines per block.
template <typename MUL>
__device__ __forceinline__ void lines_x(const Grid& g, cplx<double>* f, const double* twx, MUL mul) {
  __shared__ cplx<double> s[256];
  __shared__ double2 w[256];
  const int n = g.NLx, es = g.NLy * g.NLz, lpb = 256 / n, t = threadIdx.x;
  const int e = t / lpb, li = t - e * lpb, l = blockIdx.x * lpb + li;
  const bool ok = e < n && l < es;
  if (t < n) w[t] = make_double2(twx[2 * t], twx[2 * t + 1]);
  if (ok) s[e * lpb + li] = f[l + (size_t)e * es];
  __syncthreads();
  cplx<double> r{0, 0};
  if (ok) {
    r = line_sum(s + li, lpb, n, e, w, -1.0);
    const double m = mul(e, l / g.NLz, l % g.NLz);
    r.re *= m;
    r.im *= m;
  }
  __syncthreads();
  if (ok) s[e * lpb + li] = r;
  __syncthreads();
  if (ok) f[l + (size_t)e * es] = line_sum(s + li, lpb, n, e, w, 1.0);
}
inline int lines_x_blocks(const Grid& g) {
  const int lpb = 256 / g.NLx;
  return (g.NLy * g.NLz + lpb - 1) / lpb;
}

}  // namespace dft
}  // namespace salmon
