// Gram-Schmidt of FP64 orbitals in panels of 16 bands on the matrix cores.
//
// Band by band (k_gs_sub, k_gs_scale with k_cg_proj) each band takes five
// dependent launches that stream the finished bands for one vector: 64 bands of
// 32^3 took 5 ms, 20 times their traffic.  Here a panel P of up to 16 bands is
// orthogonalised to the finished bands Q and within itself at once, twice:
//   C = Hxyz Q^H P and G = Hxyz P^H P in one pass (k_gsb_overlap), the Cholesky
//   factor R of G - C^H C (the Gram matrix of P - Q C) in its last block, and
//   P <- (P - Q C) R^-1 = [Q P] W in one more (k_gsb_apply).
// R is upper triangular with a positive diagonal, so the result is that of the
// sequential loop (Gram_Schmidt_ompk, ARTED/GS/Gram_Schmidt.f90:41-51) up to
// rounding: the first round leaves an overlap of eps * kappa^2, the second, on
// nearly orthonormal bands, of eps.  kappa^2 = sum_ij |R^-1(i,j)|^2 |P_i|^2 is the
// squared condition of the panel, its bands scaled to norm one, against the
// finished bands: it also sees what no pivot of R shows by itself, bands that each
// keep a part of their norm but lose it in turn (b_j = e_{j-1} + e_j / 30: every
// pivot 1e-3, and twelve of them dependent to rounding).  A panel past kGsbCond, or
// one that is not finite, clears its k point's flag before it changes: the k point's
// bands stay as they are from there on, and the caller runs the band-by-band form for
// such k points.
// Up to the limit the results differ from that form's by eps * kappa, 1e-12.
//
// Per panel round that is two launches for the finished bands' bytes read twice
// and the panel's read twice and written once.  Measured, band by band and in
// panels: one Gram_Schmidt of 64 bands of 32^3 about 5 ms and 1 ms, a 64-band
// 32^3 sweep 51.9 and 46.5 ms, two sweeps of 16 bands of 16^3 at 8 k points 13.5
// and 11.5 ms, ten steps of 276 complex64 orbitals of 20x20x28 with two of them
// reorthonormalised 5.39 and 3.21 ms.
// Both passes are products of real matrices (complex as four real ones) on
// v_mfma_f64_16x16x4; their operands come straight from global memory, 64 bytes
// of a band per lane row (overlap) or 256 (apply).
#pragma once
#include "cg.hpp"

namespace salmon {
namespace cg {

constexpr int kPanel = 16;
constexpr double kGsbCond = 1e8;

struct GsBlock {
  cplx<double>* zu;     // (NK, NB, NL)
  cplx<double>* part;   // (NK, tiles, nchunk, 16, 16) partial overlaps
  cplx<double>* C;      // (NK, NB, 16) overlaps of the panel with bands 0 .. j0 + np - 1
  cplx<double>* W;      // (NK, NB, 16)
  unsigned* cnt;        // (NK, tiles + 1) arrivals, zero between launches
  int* fine;            // (NK) zero: a panel could not be orthogonalised; the k point's bands stay from there on
  int NK, NB, NL, nchunk, chunk, ntile;
  double Hxyz;
};

typedef double f64x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f64x4 mfma_f64(double a, double b, f64x4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ void store_agent(cplx<double>* p, cplx<double> v) {
  __hip_atomic_store(&p->re, v.re, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(&p->im, v.im, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ cplx<double> load_agent(const cplx<double>* p) {
  return {__hip_atomic_load(&p->re, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT),
          __hip_atomic_load(&p->im, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)};
}

// Whether this block is the last of n to arrive at *c (which returns to zero);
// all of its threads get the answer, and the others' store_agent values are visible to them.
__device__ __forceinline__ bool arrive_last(unsigned* c, unsigned n) {
  __shared__ int last;
  agent_stores_done();  // every wave's
  __syncthreads();
  if (threadIdx.x == 0) {
    last = agent_arrive(c) == n - 1;
    if (last) __hip_atomic_store(c, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  const bool l = last != 0;
  __syncthreads();
  return l;
}

// Overlaps of the panel's np bands from j0 on with bands 0 .. j0 + np - 1, and W.
// Grid (nchunk, tiles of the bands, NK), 256 threads: wave w takes every fourth
// 16 points of the chunk, lane (g, i) = (lane / 16, lane % 16) point 4 s + g.
__global__ void __launch_bounds__(256) k_gsb_overlap(GsBlock b, int j0, int np) {
  const int k = blockIdx.z, tile = blockIdx.y, c = blockIdx.x, t = threadIdx.x;
  const int lane = t & (kWave - 1), wv = t / kWave, lg = lane >> 4, li = lane & 15;
  const int nt = gridDim.y, ni = j0 + np;
  if (!b.fine[k]) return;  // (cleared by an earlier launch: all of the k point's blocks leave)
  const cplx<double>* Z = b.zu + (size_t)k * b.NB * b.NL;
  // bands past the tile's or the panel's last: its last, weighted by zero
  const int ia = tile * 16 + li, ib = j0 + li;
  const cplx<double>* A = Z + (size_t)min(ia, ni - 1) * b.NL;
  const cplx<double>* P = Z + (size_t)min(ib, ni - 1) * b.NL;
  const bool oka = ia < ni, okb = li < np;
  const int p0 = c * b.chunk, p1 = min(b.NL, p0 + b.chunk);
  f64x4 cr = {0, 0, 0, 0}, ci = cr;
  // two groups of 16 points with their loads in flight together: the loop's time
  // is their latency
  for (int q = p0 + wv * 16; q < p1; q += 128) {
    cplx<double> x[8], y[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int p = q + (s & 4) * 16 + 4 * (s & 3) + lg, pc = min(p, p1 - 1);
      x[s] = A[pc];
      y[s] = P[pc];
    }
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const bool ok = q + (s & 4) * 16 + 4 * (s & 3) + lg < p1;
      x[s].re = ok && oka ? x[s].re : 0.0;
      x[s].im = ok && oka ? x[s].im : 0.0;
      y[s].re = ok && okb ? y[s].re : 0.0;
      y[s].im = ok && okb ? y[s].im : 0.0;
    }
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      cr = mfma_f64(x[s].re, y[s].re, cr);
      ci = mfma_f64(x[s].re, y[s].im, ci);
      cr = mfma_f64(x[s].im, y[s].im, cr);
      ci = mfma_f64(-x[s].im, y[s].re, ci);
    }
  }
  // the four waves' sums, element (row lg + 4 r, column li)
  __shared__ cplx<double> red[4][256];
#pragma unroll
  for (int r = 0; r < 4; ++r) red[wv][(lg + 4 * r) * 16 + li] = cplx<double>{cr[r], ci[r]};
  __syncthreads();
  {
    cplx<double> v = red[0][t];
#pragma unroll
    for (int w = 1; w < 4; ++w) {
      v.re += red[w][t].re;
      v.im += red[w][t].im;
    }
    store_agent(&b.part[(((size_t)k * b.ntile + tile) * b.nchunk + c) * 256 + t], v);
  }
  unsigned* cnt = b.cnt + (size_t)k * (b.ntile + 1);
  if (!arrive_last(cnt + 1 + tile, b.nchunk)) return;
  // this tile's sums over the chunks, in chunk order
  {
    const cplx<double>* q = b.part + ((size_t)k * b.ntile + tile) * b.nchunk * 256 + t;
    double sr = 0.0, si = 0.0;
    for (int e0 = 0; e0 < b.nchunk; e0 += 16) {  // 16 loads in flight, clamped
      cplx<double> v[16];
#pragma unroll
      for (int e = 0; e < 16; ++e) v[e] = load_agent(q + (size_t)min(e0 + e, b.nchunk - 1) * 256);
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        sr = e0 + e < b.nchunk ? sr + v[e].re : sr;
        si = e0 + e < b.nchunk ? si + v[e].im : si;
      }
    }
    const int i = tile * 16 + t / 16;
    if (i < b.NB) store_agent(&b.C[((size_t)k * b.NB + i) * 16 + (t & 15)], cplx<double>{sr * b.Hxyz, si * b.Hxyz});
  }
  if (!arrive_last(cnt, nt)) return;
  // the last tile's block: G - C^H C, its Cholesky factor and inverse, W.  C comes
  // in tiles of 16 bands, a value per thread, the next one while one is used.
  __shared__ cplx<double> G[16][17], R[16][17], Ct[16][17];
  __shared__ double norm[16], cond[4];  // squared norms of the panel's bands before; sums of kappa^2 by wave
  const int row = t / 16, col = t & 15;
  const cplx<double>* C = b.C + (size_t)k * b.NB * 16 + row * 16 + col;
  auto next = [&](int i) { return load_agent(C + (size_t)min(i, j0 - 16) * 16); };  // (j0: whole panels)
  {
    cplx<double> v{row == col ? 1.0 : 0.0, 0.0}, ct{0, 0};
    if (j0 > 0) ct = next(0);
    if (row < np && col < np) {
      v = load_agent(C + (size_t)j0 * 16);
      if (row == col) norm[row] = v.re;
    }
    for (int i0 = 0; i0 < j0; i0 += 16) {
      Ct[row][col] = ct;
      __syncthreads();
      ct = next(i0 + 16);
      if (row < np && col < np) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const cplx<double> x = Ct[i][row], y = Ct[i][col];
          v.re -= x.re * y.re + x.im * y.im;
          v.im -= x.re * y.im - x.im * y.re;
        }
      }
      __syncthreads();
    }
    G[row][col] = v;
    R[row][col] = cplx<double>{row == col ? 1.0 : 0.0, 0.0};
  }
  __syncthreads();
  // right-looking elimination of the upper triangle; R becomes the inverse of the
  // factor: column j of R^-1 follows the same row operations from the right
  for (int j = 0; j < 16; ++j) {
    const double d = G[j][j].re;  // (not positive: infinities or NaN in R)
    const double inv = 1.0 / sqrt(d);
    const cplx<double> u{G[j][col].re * inv, G[j][col].im * inv};  // row j of the factor
    const cplx<double> l{G[j][row].re * inv, G[j][row].im * inv};
    const cplx<double> rj{R[row][j].re * inv, R[row][j].im * inv};
    __syncthreads();
    if (row > j && col > j) {  // G(row, col) -= conj(U(j, row)) U(j, col)
      G[row][col].re -= l.re * u.re + l.im * u.im;
      G[row][col].im -= l.re * u.im - l.im * u.re;
    }
    if (col == j) {
      R[row][j] = rj;
    } else if (col > j) {  // R(:, col) -= R(:, j) U(j, col)
      R[row][col].re -= rj.re * u.re - rj.im * u.im;
      R[row][col].im -= rj.re * u.im + rj.im * u.re;
    }
    __syncthreads();
  }
  {
    const cplx<double> r = R[row][col];
    const double q = wave_sum(row < np && col < np ? (r.re * r.re + r.im * r.im) * norm[row] : 0.0);
    if (lane == 0) cond[wv] = q;
  }
  __syncthreads();
  if (!((cond[0] + cond[1]) + (cond[2] + cond[3]) <= kGsbCond)) {
    if (t == 0) b.fine[k] = 0;
    return;
  }
  cplx<double>* W = b.W + (size_t)k * b.NB * 16;
  cplx<double> ct{0, 0};
  if (j0 > 0) ct = next(0);
  for (int i0 = 0; i0 < j0; i0 += 16) {  // -C R^-1
    Ct[row][col] = ct;
    __syncthreads();
    ct = next(i0 + 16);
    cplx<double> v{0, 0};
#pragma unroll
    for (int m = 0; m < 16; ++m) {
      const cplx<double> x = Ct[row][m], y = R[m][col];  // (zero for m > col)
      v.re -= x.re * y.re - x.im * y.im;
      v.im -= x.re * y.im + x.im * y.re;
    }
    W[(size_t)(i0 + row) * 16 + col] = v;
    __syncthreads();
  }
  if (row < np) W[(size_t)(j0 + row) * 16 + col] = R[row][col];
}

// P <- [Q P] W.  A wave takes 16 points: rows = panel bands, columns = points,
// four bands of [Q P] per step.  Grid (ceil(NL / 64), NK), 256 threads.
__global__ void __launch_bounds__(256) k_gsb_apply(GsBlock b, int j0, int np) {
  const int k = blockIdx.y, t = threadIdx.x;
  const int lane = t & (kWave - 1), wv = t / kWave, lg = lane >> 4, li = lane & 15;
  if (!b.fine[k]) return;
  const int p = blockIdx.x * 64 + wv * 16 + li, pc = min(p, b.NL - 1), n = j0 + np;
  cplx<double>* Z = b.zu + (size_t)k * b.NB * b.NL;
  const cplx<double>* W = b.W + (size_t)k * b.NB * 16;
  f64x4 dr = {0, 0, 0, 0}, di = dr;
#pragma unroll 4
  for (int i0 = 0; i0 < n; i0 += 4) {
    const int i = i0 + lg, ic = min(i, n - 1);
    cplx<double> w = W[(size_t)ic * 16 + li];
    const cplx<double> x = Z[(size_t)ic * b.NL + pc];
    w.re = i < n ? w.re : 0.0;
    w.im = i < n ? w.im : 0.0;
    dr = mfma_f64(w.re, x.re, dr);
    di = mfma_f64(w.re, x.im, di);
    dr = mfma_f64(-w.im, x.im, dr);
    di = mfma_f64(w.im, x.re, di);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int j = lg + 4 * r;
    if (j < np && p < b.NL) Z[(size_t)(j0 + j) * b.NL + p] = cplx<double>{dr[r], di[r]};
  }
}

}  // namespace cg
}  // namespace salmon
