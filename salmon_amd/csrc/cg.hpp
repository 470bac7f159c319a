// Ground-state kernels: the band-by-band CG of CG_ompk
// (ARTED/GS/CG.f90:34-139), the kinetic preconditioner applied to its
// residual, and the subspace matrix / rotation of diag_omp
// (ARTED/GS/diag.f90:95-130).  FP64 throughout.
//
// CG runs all k points of one band at once (grid.y = k).  Every scalar of the
// iteration (<x|H|x>, |g|^2, the 2x2 Rayleigh-Ritz coefficients, the exit
// flag) lives in device memory, so a band's whole iteration sequence is
// enqueued without a host round trip: reductions end in the last-arriving
// block of each k, which sums the per-block partials in a fixed order (so
// results do not depend on scheduling) and computes the scalar.
// A k whose band met the exit test (|ev - <x|H|x>| < 1e-15, CG.f90:114)
// skips the remaining iteration kernels.
#pragma once
#include "dft.hpp"
#include "streamed.hpp"

namespace salmon {
namespace cg {

constexpr int kPPT = 2;              // points per thread of a projection block
constexpr int kChunk = 256 * kPPT;   // points per projection block
constexpr int kJG = 8;               // lower bands per projection block
// The subtractions run in blocks of 1024 threads: every block of a k point arrives
// at one counter, and those atomics are served one by one (per launch, 32^3 and 8 k
// points of 16^3: 9.4 and 10.7 us with blocks of 64 points, 8.2 and 8.7 of 256).
constexpr int kWide = 1024;
constexpr int kSubPts = 256;  // points per subtraction block; its waves share the bands

// per-k scalars (double slots)
enum : int {
  XHX = 0, XTX, GKGK, UK, SN, EVX, CXR, CXI, CP, ZSR, ZSI, EFIN, XN, kNS = 16
};

struct State {
  double* sc;        // (NK*kNS)
  int* done;         // (NK) exit flag of the current band
  int* iters;        // (NK*NB) iterations used by each band
  double* esp_var;   // (NK*NB)
  double* part;      // (NK*maxblk*kPartQ) per-block partial sums
  unsigned* cnt;     // (NK) arrival counters of the last-block reductions
  cplx<double>* zs;  // (NK*NB) projections on the lower bands
  cplx<double>* gram;  // (NK*NB*NB) G(j,i) = Hxyz <B_j|B_i>, i < j, of the stored bands
  cplx<double>* minv;  // (NK*NB*NB) rows of (I + L)^-1, L(j,i) = G(j,i) for i < j
  double* minvr;       // (NK*NB*NB) rows of (I + Re L)^-1
  const double* occ; // (NK*NB)
  int NK, NB, NL;
  int nchunk;        // blocks of a projection (kChunk points)
  int nsub;          // blocks of a subtraction (kSubPts points)
  int nvec;          // blocks of the other kernels (256 points)
  int pstride;       // doubles of part per k
  double Hxyz;
};
constexpr int kPartQ = 2 * kJG;

// Sums NQ per-block values over the nblk blocks of row k = blockIdx.y in a fixed
// order.  Returns true in the block that arrives last; there, tot[] holds the
// totals in thread 0.  Its threads load the partials side by side: one thread
// reading them in block order took 1 to 3 us per launch on 32 to 128 blocks.
template <int NQ, int NT = 256>
__device__ bool last_block_sum(double (&v)[NQ], const State& S, int nblk, int bid, double (&tot)[NQ]) {
  constexpr int NW = NT / kWave;
  __shared__ double smem[NW * NQ];
  __shared__ int is_last;
  const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
  auto block = [&](double (&a)[NQ]) {  // valid in thread 0
#pragma unroll
    for (int q = 0; q < NQ; ++q) a[q] = wave_sum(a[q]);
    if (lane == 0) {
#pragma unroll
      for (int q = 0; q < NQ; ++q) smem[wv * NQ + q] = a[q];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
      for (int q = 0; q < NQ; ++q)
        for (int w = 1; w < NW; ++w) a[q] += smem[w * NQ + q];
    }
    __syncthreads();
  };
  block(v);
  const int k = blockIdx.y;
  double* part = S.part + (size_t)k * S.pstride;
  if (threadIdx.x == 0) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) __hip_atomic_store(&part[bid * NQ + q], v[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    agent_stores_done();
    const unsigned t = agent_arrive(&S.cnt[k]);
    is_last = (t == (unsigned)(nblk - 1));
    if (is_last) __hip_atomic_store(&S.cnt[k], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!is_last) return false;
#pragma unroll
  for (int q = 0; q < NQ; ++q) tot[q] = 0.0;
  for (int b = threadIdx.x; b < nblk; b += NT) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) tot[q] += __hip_atomic_load(&part[b * NQ + q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  block(tot);
  return true;
}

// Keeps the loads of v before this point.  The kernels look at the exit flag
// after their loads, so that it does not add a memory round trip to each launch.
__device__ __forceinline__ void loaded(const cplx<double>& v) { asm volatile("" ::"v"(v.re), "v"(v.im)); }

__device__ __forceinline__ cplx<double> cmulc(cplx<double> a, cplx<double> b) {  // a*b
  return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}

// Source vector of the projection and subtraction kernels: either a stored
// vector V, or the residual H x - <x|H|x> x formed on the fly (CG.f90:85).
struct Src {
  const cplx<double>* v;   // stored vector (nullptr: residual)
  size_t vstride;          // distance between the vectors of consecutive k
  const cplx<double>* hx;  // residual operands, NL apart per k
  const cplx<double>* x;
  __device__ __forceinline__ cplx<double> at(int k, int NL, int p, double xhx) const {
    if (v) return v[(size_t)k * vstride + p];
    const size_t o = (size_t)k * NL + p;
    const cplx<double> h = hx[o], e = x[o];
    return {h.re - xhx * e.re, h.im - xhx * e.im};
  }
};

// Projections on the lower bands.  The reference orthogonalises with the
// sequential (modified) Gram-Schmidt loop (CG.f90:69-71, 86-89): the
// coefficient of band j is taken against the vector already stripped of bands
// 0..j-1.  Its coefficients c solve c_j = b_j - sum_{k<j} G_jk c_k with
// b_j = Hxyz <B_j|v> and the Gram matrix G_jk = Hxyz <B_j|B_k> of the lower
// bands, which the lower bands need not make diagonal (the start vector's
// overlap keeps only its real part, CG.f90:46,70, so a band may keep an
// imaginary overlap with the bands below it).  k_cg_proj forms b in one
// parallel pass and solves the triangle in the last block, as c = M b with
// M = (I + L)^-1 (L the strictly lower part of G): G does not change while a
// band iterates, so M gains one row per stored band and each solve is a
// parallel matrix-vector product instead of ib dependent steps.
//   PROJ_START  real coefficients (real(8) :: s, CG.f90:46,70): the
//               recurrence keeps c real, so c = (I + Re L)^-1 Re b
//   PROJ_VEC    complex coefficients (CG.f90:86-89)
//   PROJ_GRAM   stores row ib of G from the stored band ib, and row ib of
//               both inverses: M(ib, l) = -sum_{l<=q<ib} G(ib, q) M(q, l)
//               (unit diagonal implicit).
//   PROJ_PLAIN  b itself (Gram-Schmidt).
// ib is at most kCgMaxNB (PROJ_PLAIN takes more lower bands in several launches).
// Grid: (nchunk, ceil(ib/kJG), NK).
enum : int { PROJ_START = 0, PROJ_VEC = 1, PROJ_GRAM = 2, PROJ_PLAIN = 3 };
constexpr int kCgMaxNB = 1024;

__global__ void __launch_bounds__(256) k_cg_proj(State S, const cplx<double>* __restrict__ zu, int ib, Src src,
                                                 int mode, int check_done) {
  const int k = blockIdx.z;
  const int skip = check_done ? S.done[k] : 0;
  const int t = threadIdx.x, c = blockIdx.x, g0 = blockIdx.y * kJG;
  const int nj = min(kJG, ib - g0);
  const double xhx = S.sc[k * kNS + XHX];
  const cplx<double>* B = zu + (size_t)k * S.NB * S.NL;
  double acc[2 * kJG];
#pragma unroll
  for (int q = 0; q < 2 * kJG; ++q) acc[q] = 0.0;
  // every load of the block is unconditional (points past the grid read
  // point 0, bands past ib the last lower band; their terms are zeroed by a
  // select), so no branch separates the loads from their uses and they are
  // in flight together; each band's sum takes its points in the same order
  cplx<double> e[kPPT];
  int pc[kPPT];
  bool okp[kPPT];
#pragma unroll
  for (int i = 0; i < kPPT; ++i) {
    const int p = c * kChunk + i * 256 + t;
    okp[i] = p < S.NL;
    pc[i] = okp[i] ? p : 0;
  }
  // (Src::at with its source choice outside the point loop)
  if (src.v) {
#pragma unroll
    for (int i = 0; i < kPPT; ++i) e[i] = src.v[(size_t)k * src.vstride + pc[i]];
  } else {
#pragma unroll
    for (int i = 0; i < kPPT; ++i) e[i] = src.at(k, S.NL, pc[i], xhx);
  }
#pragma unroll
  for (int j = 0; j < kJG; ++j) {
    const int jb = min(g0 + j, ib - 1);
#pragma unroll
    for (int i = 0; i < kPPT; ++i) {
      const cplx<double> b0 = B[(size_t)jb * S.NL + pc[i]];
      const bool w = okp[i] && j < nj;
      const double br = w ? b0.re : 0.0, bi = w ? b0.im : 0.0;
      acc[2 * j] += br * e[i].re + bi * e[i].im;
      acc[2 * j + 1] += br * e[i].im - bi * e[i].re;
    }
  }
  loaded(cplx<double>{acc[0], acc[2 * kJG - 1]});
  if (skip) return;
  // partials: [chunk][group][2*kJG]
  __shared__ double smem[256];
  __shared__ int is_last;
  const int lane = t & (kWave - 1), wv = t / kWave, np = gridDim.y * kPartQ;
  wave_sums(acc);
#pragma unroll
  for (int q = 0; q < kPartQ; ++q)
    if (lane == wave_sums_lane(q)) smem[wv * kPartQ + q] = acc[0];
  double* part = S.part + (size_t)k * S.pstride;
  __syncthreads();
  if (t < kPartQ) {
    const double v = (smem[t] + smem[kPartQ + t]) + (smem[2 * kPartQ + t] + smem[3 * kPartQ + t]);
    __hip_atomic_store(&part[(size_t)c * np + blockIdx.y * kPartQ + t], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    agent_stores_done();
  }
  if (t == 0) {  // (in the wave that stored)
    is_last = agent_arrive(&S.cnt[k]) == gridDim.x * gridDim.y - 1;
    if (is_last) __hip_atomic_store(&S.cnt[k], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!is_last) return;
  // The last block of row k, which the launch waits for: its loads are few rounds
  // of many in flight.  The first of the inverse's rows, which do not depend on the
  // sums, come with them: four threads (quad qd, part qi) per row, each every
  // fourth column.
  cplx<double>* gram = S.gram + (size_t)k * S.NB * S.NB;
  cplx<double>* M = S.minv + (size_t)k * S.NB * S.NB;
  double* MR = S.minvr + (size_t)k * S.NB * S.NB;
  constexpr int kTail = 16;
  const int qd = t >> 2, qi = t & 3;
  cplx<double> mm[kTail];
  auto row = [&](int j0, int l0) {  // M(j0 + qd, l0 + qi + 4 u), l < j; clamped elsewhere
    const int j = min(j0 + qd, ib - 1);
#pragma unroll
    for (int u = 0; u < kTail; ++u) {
      const size_t o = (size_t)j * S.NB + min(l0 + qi + 4 * u, j);
      if (mode == PROJ_START) mm[u] = cplx<double>{MR[o], 0.0};
      else mm[u] = M[o];
    }
  };
  if (mode == PROJ_START || mode == PROJ_VEC) row(0, 0);
  // sums over the chunks: thread (value, share of the chunks), then the shares in order
  __shared__ cplx<double> zsh[kCgMaxNB];
  double* zv = (double*)zsh;
  int lg = 0;
  while ((1 << lg) < 2 * ib && lg < 8) ++lg;
  const int nv = 1 << lg, ns = 256 >> lg, sh = t >> lg;
  for (int v0 = 0; v0 < 2 * ib; v0 += nv) {
    const int v = v0 + (t & (nv - 1)), vc = min(v, 2 * ib - 1);
    double s = 0.0;
    for (int c0 = sh; c0 < S.nchunk; c0 += 8 * ns) {
      double a[8];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        a[u] = __hip_atomic_load(&part[(size_t)min(c0 + u * ns, S.nchunk - 1) * np + vc], __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
      for (int u = 0; u < 8; ++u) s = c0 + u * ns < S.nchunk ? s + a[u] : s;
    }
    __syncthreads();
    smem[t] = s;
    __syncthreads();
    if (sh == 0 && v < 2 * ib) {
      for (int r = 1; r < ns; ++r) s += smem[r * nv + t];
      zv[v] = s * S.Hxyz;
    }
  }
  __syncthreads();
  if (mode == PROJ_PLAIN) {  // coefficients against the unmodified vector
    for (int j = t; j < ib; j += 256) S.zs[(size_t)k * S.NB + j] = zsh[j];
    return;
  }
  auto quad = [](double v) {
    v += dpp_mov<dpp::kQuad1032, 0xf>(v);
    return v + dpp_mov<dpp::kQuad2301, 0xf>(v);
  };
  if (mode == PROJ_GRAM) {
    // raw_j = Hxyz <B_j|B_ib>, so G(ib, j) = conj(raw_j)
    for (int j = t; j < ib; j += 256) gram[(size_t)ib * S.NB + j] = cplx<double>{zsh[j].re, -zsh[j].im};
    // the unit diagonal of M is implicit (band 0 has no projection launch)
    for (int j0 = 0; j0 < ib; j0 += 64) {
      const int l = j0 + qd, lc = min(l, ib - 1);
      double sr = 0.0, si = 0.0, rr = 0.0;
      if (qi == 0) {  // q = l: G(ib, l) M(l, l)
        sr = rr = zsh[lc].re;
        si = -zsh[lc].im;
      }
      for (int q0 = j0 + qi; q0 < ib; q0 += 4 * kTail) {
        double mr[kTail];
#pragma unroll
        for (int u = 0; u < kTail; ++u) {
          const size_t o = (size_t)max(min(q0 + 4 * u, ib - 1), lc) * S.NB + lc;  // (row q > column l, or not used)
          mm[u] = M[o];
          mr[u] = MR[o];
        }
#pragma unroll
        for (int u = 0; u < kTail; ++u) {
          const int q = q0 + 4 * u;
          const bool ok = q > l && q < ib;
          const cplx<double> z = zsh[min(q, ib - 1)];
          sr = ok ? sr + (z.re * mm[u].re + z.im * mm[u].im) : sr;
          si = ok ? si + (z.re * mm[u].im - z.im * mm[u].re) : si;
          rr = ok ? rr + z.re * mr[u] : rr;
        }
      }
      sr = quad(sr);
      si = quad(si);
      rr = quad(rr);
      if (qi == 0 && l < ib) {
        M[(size_t)ib * S.NB + l] = cplx<double>{-sr, -si};
        MR[(size_t)ib * S.NB + l] = -rr;
      }
    }
    return;
  }
  // c = M b (PROJ_START: of the real parts)
  const bool real = mode == PROJ_START;
  for (int j0 = 0; j0 < ib; j0 += 64) {
    const int j = min(j0 + qd, ib - 1);
    double cr = qi == 0 ? zsh[j].re : 0.0, ci = qi == 0 && !real ? zsh[j].im : 0.0;
    for (int l0 = 0; l0 < min(ib, j0 + 64); l0 += 4 * kTail) {
      if (j0 > 0 || l0 > 0) row(j0, l0);
#pragma unroll
      for (int u = 0; u < kTail; ++u) {
        const int l = l0 + qi + 4 * u;
        const cplx<double> m = mm[u], z = zsh[min(l, j)];
        const double zi = real ? 0.0 : z.im;
        cr = l < j ? cr + (m.re * z.re - m.im * zi) : cr;
        ci = l < j ? ci + (m.re * zi + m.im * z.re) : ci;
      }
    }
    cr = quad(cr);
    ci = quad(ci);
    if (qi == 0 && j0 + qd < ib) S.zs[(size_t)k * S.NB + j] = cplx<double>{cr, ci};
  }
}

// Roles of the subtraction kernel's reduction.
enum : int {
  SUB_START = 0,  // start vector: SN = 1/sqrt(|out|^2 Hxyz); resets the band's flags
  SUB_GRAD = 1,   // residual, no preconditioner: s = |g|^2 Hxyz (CG.f90:90)
  SUB_PCDIR = 2,  // preconditioned residual: s = Re<Kg|g> Hxyz
  SUB_NONE = 3,   // no reduction
  SUB_LEARN = 4   // learned direction: no conjugation (uk = 0); the network is
                  // not a fixed linear operator, so each iteration is a
                  // preconditioned steepest-descent step with the 2x2 Rayleigh-Ritz
};

// out = src - sum_{j<ib} zs(j) B_j  (CG.f90:69-71, 86-89), then the role's
// reduction.  For a search direction d (the roles but SUB_START and SUB_NONE) the
// finisher forms the conjugation ratio uk = s/gkgk (CG.f90:92-98; iteration 1
// takes p = d) and, from <x|d> and <x|p_old>, the overlap zs = <x|d + uk p_old>
// that the direction is stripped of (CG.f90:103), so p needs no pass of its own.
// Each quarter of a block takes every fourth band for the block's points, whose
// sum the first quarter forms: the loop's loads are the launch's time (64 bands:
// 8 loads in flight per lane, two rounds of them instead of eight).
// Grid (nsub, NK), kWide threads.
__global__ void __launch_bounds__(kWide) k_cg_sub(State S, const cplx<double>* __restrict__ zu, int ib, Src src,
                                                cplx<double>* out, const cplx<double>* __restrict__ other,
                                                const cplx<double>* __restrict__ x, const cplx<double>* __restrict__ P,
                                                int role, int it, int ncg) {
  const int k = blockIdx.y;
  const int skip = role != SUB_START ? S.done[k] : 0;
  // consecutive blocks go to consecutive ones of the eight dies: the die of a
  // projection block's kChunk points also takes the two blocks here that hold them,
  // and finds the lower bands in its L2 cache
  int c = blockIdx.x;
  if ((c | 15) < S.nsub) c = (c & ~15) | (c & 7) << 1 | (c >> 3 & 1);
  const int t = threadIdx.x & (kSubPts - 1);
  const int part = __builtin_amdgcn_readfirstlane(threadIdx.x / kSubPts);
  static_assert(kChunk == 2 * kSubPts, "two subtraction blocks per projection block");
  const size_t off = (size_t)k * S.NL;
  const double xhx = S.sc[k * kNS + XHX];
  const cplx<double>* B = zu + (size_t)k * S.NB * S.NL;
  const cplx<double>* zs = S.zs + (size_t)k * S.NB;
  const int p = c * kSubPts + t, pc = min(p, S.NL - 1);
  const bool dir = role != SUB_START && role != SUB_NONE;
  cplx<double> e{0, 0}, o{0, 0}, xp{0, 0}, q{0, 0};
  if (part == 0) {
    e = src.at(k, S.NL, pc, xhx);
    if (role == SUB_PCDIR) o = other[off + pc];
    if (dir) xp = x[off + pc];
    if (dir && it > 1 && role != SUB_LEARN) q = P[off + pc];
  }
#pragma unroll 8
  for (int j = part; j < ib; j += 4) {
    const cplx<double> b = B[(size_t)j * S.NL + pc], z = zs[j];
    e.re -= b.re * z.re - b.im * z.im;
    e.im -= b.re * z.im + b.im * z.re;
  }
  loaded(e);
  if (skip) return;
  __shared__ cplx<double> sh[3][kSubPts];
  if (part > 0) sh[part - 1][t] = e;
  __syncthreads();
  double v[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
  if (part == 0 && p < S.NL) {
#pragma unroll
    for (int w = 0; w < 3; ++w) {
      e.re += sh[w][t].re;
      e.im += sh[w][t].im;
    }
    out[off + p] = e;
    v[0] = role == SUB_PCDIR ? e.re * o.re + e.im * o.im : e.re * e.re + e.im * e.im;
    v[1] = xp.re * e.re + xp.im * e.im;
    v[2] = xp.re * e.im - xp.im * e.re;
    v[3] = xp.re * q.re + xp.im * q.im;
    v[4] = xp.re * q.im - xp.im * q.re;
  }
  if (role == SUB_NONE) return;
  double tot[5];
  if (!last_block_sum<5, kWide>(v, S, S.nsub, c, tot)) return;
  if (threadIdx.x != 0) return;
  double* sc = S.sc + k * kNS;
  if (role == SUB_START) {
    sc[SN] = 1.0 / sqrt(tot[0] * S.Hxyz);
    S.done[k] = 0;
    S.iters[(size_t)k * S.NB + ib] = ncg;
    return;
  }
  double uk = 0.0;
  if (role != SUB_LEARN) {
    const double s = tot[0] * S.Hxyz;
    if (it > 1) uk = s / sc[GKGK];
    sc[GKGK] = s;
  }
  sc[UK] = uk;
  sc[ZSR] = (uk != 0.0 ? tot[1] + uk * tot[3] : tot[1]) * S.Hxyz;
  sc[ZSI] = (uk != 0.0 ? tot[2] + uk * tot[4] : tot[2]) * S.Hxyz;
}

// p = d + uk p (CG.f90:92-98), o = p - x zs, SN = 1/sqrt(|o|^2 Hxyz)
// (CG.f90:103-105).  o stays as it is: the H application and the rotation take
// SN with it.  Grid (nvec, NK).
__global__ void __launch_bounds__(256) k_cg_pko(State S, const cplx<double>* __restrict__ d, cplx<double>* __restrict__ P,
                                                const cplx<double>* __restrict__ x, cplx<double>* __restrict__ pko) {
  const int k = blockIdx.y, c = blockIdx.x;
  const int skip = S.done[k];
  const double* sc = S.sc + k * kNS;
  const double uk = sc[UK];
  const cplx<double> z{sc[ZSR], sc[ZSI]};
  const int p = c * 256 + threadIdx.x;
  const size_t i = (size_t)k * S.NL + min(p, S.NL - 1);
  const cplx<double> e = x[i], b = P[i];  // (P holds no numbers yet at uk = 0)
  cplx<double> q = d[i];
  loaded(e);
  loaded(b);
  loaded(q);
  if (skip) return;
  double v[1] = {0.0};
  if (p < S.NL) {
    if (uk != 0.0) {
      q.re += uk * b.re;
      q.im += uk * b.im;
    }
    P[i] = q;
    q.re -= e.re * z.re - e.im * z.im;
    q.im -= e.re * z.im + e.im * z.re;
    pko[i] = q;
    v[0] = q.re * q.re + q.im * q.im;
  }
  double tot[1];
  if (!last_block_sum<1>(v, S, S.nvec, c, tot)) return;
  if (threadIdx.x == 0) S.sc[k * kNS + SN] = 1.0 / sqrt(tot[0] * S.Hxyz);
}

// KB projections of the CG's vector and the term each sphere point adds
// (pseudo_pt, ARTED/common/hpsi.f90:183-206), an atom per block:
//   U(l) = Hxyz iuV(l) sum_j uV(j,l) e^{ik.r_j} v(J_j),  dps(j) = e^{-ik.r_j} sum_l uV(j,l) U(l)
// so that the stencil pass reads one term per sphere point instead of four
// projectors' tables and a sincos each: the two launches took 15 and 6 us on
// 32^3 with 27 atoms.  A wave per projector, then a thread per point.  Grid (NI, NK).
__global__ void __launch_bounds__(256) k_cg_kb(State S, const cplx<double>* __restrict__ in, KBTables kb,
                                               const cplx<double>* __restrict__ ph, cplx<double>* __restrict__ dps,
                                               int check_done) {
  const int a = blockIdx.x, k = blockIdx.y;
  const int skip = check_done ? S.done[k] : 0;
  const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
  const int j0 = kb.atom_start[a], m = kb.atom_start[a + 1] - j0;
  const cplx<double>* E = in + (size_t)k * S.NL;
  const cplx<double>* pk = ph + (size_t)k * kb.NPI + j0;
  cplx<double>* dk = dps + (size_t)k * kb.NPI + j0;
  constexpr int kPass = 16;
  __shared__ cplx<double> U[kPass];
  const int lb = kb.atom_lma[a], le = kb.atom_lma[a + 1];
  for (int l0 = lb; l0 < le; l0 += kPass) {
    const int nl = min(kPass, le - l0);
    for (int l = wv; l < nl; l += 4) {
      const double* uv = kb.uv + (size_t)(l0 + l) * kb.Nps;
      double sr = 0.0, si = 0.0;
      // three chunks with their loads in flight; indices past the sphere: its first point, weight zero
      for (int jb = 0; jb < m; jb += 3 * kWave) {
        cplx<double> e[3], f[3];
        double u[3];
#pragma unroll
        for (int h = 0; h < 3; ++h) {
          const int j = jb + h * kWave + lane, jc = j < m ? j : 0;
          e[h] = E[kb.pidx[j0 + jc]];
          f[h] = pk[jc];
          u[h] = uv[jc];
          u[h] = j < m ? u[h] : 0.0;
        }
#pragma unroll
        for (int h = 0; h < 3; ++h) {
          sr += u[h] * (f[h].re * e[h].re - f[h].im * e[h].im);
          si += u[h] * (f[h].re * e[h].im + f[h].im * e[h].re);
        }
      }
      sr = wave_sum(sr);
      si = wave_sum(si);
      const double f = S.Hxyz * kb.lma_sign[l0 + l];
      if (lane == 0) U[l] = cplx<double>{sr * f, si * f};
    }
    __syncthreads();
    if (skip) return;
    for (int j = threadIdx.x; j < m; j += 256) {
      cplx<double> t{0, 0};
      for (int l = 0; l < nl; ++l) {
        const double u = kb.uv[(size_t)(l0 + l) * kb.Nps + j];
        t.re += u * U[l].re;
        t.im += u * U[l].im;
      }
      const cplx<double> f = pk[j];
      cplx<double> r{f.re * t.re + f.im * t.im, f.re * t.im - f.im * t.re};  // conj(f) t
      if (l0 > lb) {
        r.re += dk[j].re;
        r.im += dk[j].im;
      }
      dk[j] = r;
    }
    __syncthreads();
  }
}

// What an H application of the CG ends with.
enum : int {
  H_START = 0,  // start vector: x = s v; <x|H|x>, <x|T|x> (CG.f90:79-80), |x|^2
  H_RR = 1,     // search direction q = s o: 2x2 Rayleigh-Ritz of span{x, q} (CG.f90:107-114)
  H_EFIN = 2    // stored band = s x: e = <x|H|x> (CG.f90:122-125)
};

// h = s H v, t = s T v (nullable: only the kinetic preconditioner reads <x|T|x>)
// of the vector v, s = 1/|v|, with the KB terms of k_cg_kb; the scaled vector
// itself for H_START and H_EFIN; then the role's sums, whose operands it has at
// hand.  Grid (nvec, NK).
template <int ROLE>
__global__ void __launch_bounds__(256) k_cg_h(State S, const cplx<double>* __restrict__ v, const double* __restrict__ kac,
                                              const double* __restrict__ vloc, Grid g, KBTables kb,
                                              const cplx<double>* __restrict__ dps, cplx<double>* __restrict__ hv,
                                              cplx<double>* __restrict__ tv, cplx<double>* __restrict__ xo, size_t xstride,
                                              const cplx<double>* __restrict__ x, int ib, int it) {
  const int k = blockIdx.y, c = blockIdx.x;
  const int skip = ROLE == H_RR ? S.done[k] : 0;
  double* sc = S.sc + k * kNS;
  const int p = c * 256 + threadIdx.x, pc = min(p, S.NL - 1);
  const double s = sc[ROLE == H_EFIN ? XN : SN];
  double sum[3] = {0.0, 0.0, 0.0};
  const size_t i = (size_t)k * S.NL + pc;
  const int tp = kb.pt2t[pc];
  cplx<double> xp{0, 0};
  if (ROLE == H_RR) xp = x[i];
  double kx, ky, kz;
  orbital_k(kac, S.NK, k, 0, 0, 0, kx, ky, kz);
  cplx<double> e, t;
  double V;
  cplx<double> f = stencil_point<double>(v + (size_t)k * S.NL, pc, kx, ky, kz, vloc, g, e, V);
  loaded(f);
  loaded(xp);
  if (ROLE == H_RR && skip) return;  // the whole block, threads past the grid among them: barriers follow
  if (p < S.NL) {
    if (tv) t = cplx<double>{f.re - V * e.re, f.im - V * e.im};
    if (tp >= 0) {
      const cplx<double>* d = dps + (size_t)k * kb.NPI;
      for (int q = kb.tj_start[tp]; q < kb.tj_start[tp + 1]; ++q) {
        const cplx<double> a = d[kb.tj[q]];
        f.re += a.re;
        f.im += a.im;
      }
    }
    f.re *= s;
    f.im *= s;
    e.re *= s;
    e.im *= s;
    hv[i] = f;
    if (ROLE != H_RR) xo[(size_t)k * xstride + p] = e;
    if (tv) {
      t.re *= s;
      t.im *= s;
      tv[i] = t;
    }
    if (ROLE == H_RR) {
      sum[0] = xp.re * f.re + xp.im * f.im;
      sum[1] = xp.re * f.im - xp.im * f.re;
      sum[2] = e.re * f.re + e.im * f.im;
    } else {
      sum[0] = e.re * f.re + e.im * f.im;
      if (ROLE == H_START) {
        if (tv) sum[1] = e.re * t.re + e.im * t.im;
        sum[2] = e.re * e.re + e.im * e.im;
      }
    }
  }
  double tot[3];
  if (!last_block_sum<3>(sum, S, S.nvec, c, tot)) return;
  if (threadIdx.x != 0) return;
  if (ROLE == H_EFIN) {
    sc[EFIN] = tot[0] * S.Hxyz;
  } else if (ROLE == H_START) {
    sc[XHX] = tot[0] * S.Hxyz;
    sc[XTX] = tot[1] * S.Hxyz;
    sc[XN] = 1.0 / sqrt(tot[2] * S.Hxyz);
  } else {
    const double xhx = sc[XHX];
    const double xhp_r = tot[0] * S.Hxyz, xhp_i = tot[1] * S.Hxyz, php = tot[2] * S.Hxyz;
    const double a2 = xhp_r * xhp_r + xhp_i * xhp_i;
    const double ev = 0.5 * ((xhx + php) - sqrt((xhx - php) * (xhx - php) + 4.0 * a2));
    double cxr = xhp_r / (ev - xhx), cxi = xhp_i / (ev - xhx);
    const double cp = 1.0 / sqrt(1.0 + (cxr * cxr + cxi * cxi));
    cxr *= cp;
    cxi *= cp;
    sc[EVX] = ev;
    sc[CXR] = cxr;
    sc[CXI] = cxi;
    sc[CP] = cp;
    if (fabs(ev - xhx) < 1e-15) {
      S.done[k] = 1;
      S.iters[(size_t)k * S.NB + ib] = it;
    }
  }
}

// x = cx x + cp q, q = SN pko; hx and (nullable) tx likewise (CG.f90:115-117);
// then <x|H|x>, <x|T|x> (CG.f90:118-119) and 1/|x| for the stored band
// (CG.f90:122).  Grid (nvec, NK).
__global__ void __launch_bounds__(256) k_cg_rotate(State S, cplx<double>* __restrict__ x, cplx<double>* __restrict__ hx,
                                                   cplx<double>* __restrict__ tx, const cplx<double>* __restrict__ pko,
                                                   const cplx<double>* __restrict__ hp, const cplx<double>* __restrict__ tp) {
  const int k = blockIdx.y, c = blockIdx.x;
  const int skip = S.done[k];
  const double* sc = S.sc + k * kNS;
  const cplx<double> cx{sc[CXR], sc[CXI]};
  const double cp = sc[CP], sn = sc[SN];
  const int p = c * 256 + threadIdx.x;
  const size_t i = (size_t)k * S.NL + min(p, S.NL - 1);
  cplx<double> e = x[i], h = hx[i];
  const cplx<double> q = pko[i], hq = hp[i];
  loaded(e);
  loaded(h);
  loaded(q);
  loaded(hq);
  if (skip) return;
  double v[3] = {0.0, 0.0, 0.0};
  if (p < S.NL) {
    e = cmulc(cx, e);
    h = cmulc(cx, h);
    e.re += cp * (sn * q.re);
    e.im += cp * (sn * q.im);
    h.re += cp * hq.re;
    h.im += cp * hq.im;
    x[i] = e;
    hx[i] = h;
    v[0] = e.re * h.re + e.im * h.im;
    v[2] = e.re * e.re + e.im * e.im;
    if (tx) {
      cplx<double> t = cmulc(cx, tx[i]);
      const cplx<double> tq = tp[i];
      t.re += cp * tq.re;
      t.im += cp * tq.im;
      tx[i] = t;
      v[1] = e.re * t.re + e.im * t.im;
    }
  }
  double tot[3];
  if (!last_block_sum<3>(v, S, S.nvec, c, tot)) return;
  if (threadIdx.x == 0) {
    S.sc[k * kNS + XHX] = tot[0] * S.Hxyz;
    S.sc[k * kNS + XTX] = tot[1] * S.Hxyz;
    S.sc[k * kNS + XN] = 1.0 / sqrt(tot[2] * S.Hxyz);
  }
}

// esp_var(ib,k) = sqrt(|Hx - e x|^2 Hxyz) occ(ib,k) of the stored band x
// (CG.f90:126).  Grid (nvec, NK).
__global__ void __launch_bounds__(256) k_cg_resid(State S, const cplx<double>* __restrict__ x, size_t xstride,
                                                  const cplx<double>* __restrict__ hp, int ib) {
  const int k = blockIdx.y, c = blockIdx.x;
  const double e = S.sc[k * kNS + EFIN];
  const int p = c * 256 + threadIdx.x;
  double v[1] = {0.0};
  if (p < S.NL) {
    const cplx<double> a = x[(size_t)k * xstride + p], h = hp[(size_t)k * S.NL + p];
    const double r = h.re - e * a.re, q = h.im - e * a.im;
    v[0] = r * r + q * q;
  }
  double tot[1];
  if (!last_block_sum<1>(v, S, S.nvec, c, tot)) return;
  if (threadIdx.x == 0) {
    const size_t o = (size_t)k * S.NB + ib;
    S.esp_var[o] = sqrt(tot[0] * S.Hxyz) * S.occ[o];
  }
}

// ---------------------------------------------------------------------------
// Kinetic preconditioner K g = F^-1 [ k(x) F g ], x = t(q)/<x|T|x>, with t(q)
// the finite-difference kinetic symbol -1/2 sum_axes (lap0 + 2 sum_m lap_m
// cos(m q h)) and k(x) = f/(f + 16 x^4), f = 27 + 18x + 12x^2 + 8x^3 (the
// Teter-Payne-Allan form), in the three launches of dft.hpp (a pass per axis, five
// launches, took 30 us on 32^3).  No reference counterpart: CG_ompk applies no
// preconditioner (CG.f90:85-92).  Twiddles (cos, sin)(2 pi j/n) of axis a at
// tw + 2 * kDftMax * a, symbols at symb + kDftMax * a.
// ---------------------------------------------------------------------------
constexpr int kDftMax = 64;

// Grid (blocks of z lines, NLx, NK).
__global__ void __launch_bounds__(256) k_kin_zy(State S, const cplx<double>* __restrict__ in, cplx<double>* __restrict__ out,
                                                Grid g, int nl, const double* __restrict__ tw) {
  const int k = blockIdx.z;
  if (S.done[k]) return;
  const size_t o = (size_t)k * g.NL + (size_t)blockIdx.y * g.NLy * g.NLz;
  dft::plane<true>(g.NLz, g.NLy, nl, tw + 4 * kDftMax, tw + 2 * kDftMax, -1.0,
                   [&](int z, int y) { return in[o + y * g.NLz + z]; },
                   [&](int z, int y, cplx<double> v) { out[o + y * g.NLz + z] = v; });
}

// Grid (blocks of x lines, NK).
__global__ void __launch_bounds__(256) k_kin_x(State S, cplx<double>* __restrict__ f, Grid g, const double* __restrict__ tw,
                                               const double* __restrict__ symb) {
  const int k = blockIdx.y;
  if (S.done[k]) return;
  double txx = S.sc[k * kNS + XTX];
  if (!(txx > 1e-12)) txx = 1e-12;
  dft::lines_x(g, f + (size_t)k * g.NL, tw, [&](int ix, int iy, int iz) {
    const double x = ((symb[ix] + symb[kDftMax + iy]) + symb[2 * kDftMax + iz]) / txx;
    const double q = 27.0 + 18.0 * x + 12.0 * x * x + 8.0 * x * x * x;
    return q / (q + 16.0 * x * x * x * x) / g.NL;
  });
}

// Grid (blocks of y lines, NLx, NK).
__global__ void __launch_bounds__(256) k_kin_yz(State S, const cplx<double>* __restrict__ in, cplx<double>* __restrict__ out,
                                                Grid g, int nl, const double* __restrict__ tw) {
  const int k = blockIdx.z;
  if (S.done[k]) return;
  const size_t o = (size_t)k * g.NL + (size_t)blockIdx.y * g.NLy * g.NLz;
  dft::plane<false>(g.NLy, g.NLz, nl, tw + 2 * kDftMax, tw + 4 * kDftMax, 1.0,
                    [&](int y, int z) { return in[o + y * g.NLz + z]; },
                    [&](int y, int z, cplx<double> v) { out[o + y * g.NLz + z] = v; });
}

// ---------------------------------------------------------------------------
// Subspace matrix and rotation of diag_omp (ARTED/GS/diag.f90:111-127).
// ---------------------------------------------------------------------------

// M(i,j) partials = sum_p conj(A_i(p)) B_j(p) over a slice of points; 16x16
// tiles of (i, j), one thread per pair, points staged through LDS.
// Grid (ceil(NB/16)^2, nslice, NK); out: part[(k*nslice + slice)*NB*NB + i*NB + j].
constexpr int kTile = 16, kSlicePts = 64;
__global__ void __launch_bounds__(256) k_sub_matrix(const cplx<double>* __restrict__ A, const cplx<double>* __restrict__ B,
                                                    int NB, int NL, int pts_per_slice, double* __restrict__ part) {
  const int ntile = (NB + kTile - 1) / kTile;
  const int ti = blockIdx.x / ntile, tj = blockIdx.x % ntile;
  const int k = blockIdx.z, slice = blockIdx.y, nslice = gridDim.y;
  const int i = ti * kTile + threadIdx.x / kTile, j = tj * kTile + threadIdx.x % kTile;
  __shared__ cplx<double> sa[kTile][kSlicePts + 1], sb[kTile][kSlicePts + 1];
  const cplx<double>* Ak = A + (size_t)k * NB * NL;
  const cplx<double>* Bk = B + (size_t)k * NB * NL;
  const int p0 = slice * pts_per_slice, p1 = min(NL, p0 + pts_per_slice);
  double re = 0.0, im = 0.0;
  for (int q0 = p0; q0 < p1; q0 += kSlicePts) {
    for (int idx = threadIdx.x; idx < kTile * kSlicePts; idx += 256) {
      const int r = idx / kSlicePts, pp = idx % kSlicePts, p = q0 + pp;
      const int ia = ti * kTile + r, jb = tj * kTile + r;
      sa[r][pp] = (ia < NB && p < p1) ? Ak[(size_t)ia * NL + p] : cplx<double>{0.0, 0.0};
      sb[r][pp] = (jb < NB && p < p1) ? Bk[(size_t)jb * NL + p] : cplx<double>{0.0, 0.0};
    }
    __syncthreads();
    const int r = threadIdx.x / kTile, cc = threadIdx.x % kTile;
#pragma unroll 8
    for (int pp = 0; pp < kSlicePts; ++pp) {
      const cplx<double> a = sa[r][pp], b = sb[cc][pp];
      re += a.re * b.re + a.im * b.im;
      im += a.re * b.im - a.im * b.re;
    }
    __syncthreads();
  }
  if (i < NB && j < NB) {
    double* o = part + ((size_t)k * nslice + slice) * NB * NB * 2;
    o[2 * ((size_t)i * NB + j)] = re;
    o[2 * ((size_t)i * NB + j) + 1] = im;
  }
}

// sums the slices in order: M(k, i, j) * scale
__global__ void __launch_bounds__(256) k_sub_matrix_sum(const double* __restrict__ part, int NB, int nslice,
                                                        double scale, double* __restrict__ M) {
  const int k = blockIdx.y;
  const int idx = blockIdx.x * 256 + threadIdx.x;
  if (idx >= NB * NB * 2) return;
  double s = 0.0;
#pragma unroll 8
  for (int sl = 0; sl < nslice; ++sl) s += part[((size_t)k * nslice + sl) * NB * NB * 2 + idx];
  M[(size_t)k * NB * NB * 2 + idx] = s * scale;
}

// C_i(p) = sum_j A_j(p) U(j, i) for 16 outputs i per thread (U column-major
// per k: U[(k*NB + i)*NB + j]).  Grid (ceil(NL/256), ceil(NB/16), NK).
__global__ void __launch_bounds__(256) k_rotate_bands(const cplx<double>* __restrict__ A, const cplx<double>* __restrict__ U,
                                                     cplx<double>* __restrict__ C, int NB, int NL) {
  const int k = blockIdx.z, i0 = blockIdx.y * kTile;
  const int p = blockIdx.x * 256 + threadIdx.x;
  extern __shared__ cplx<double> su[];  // NB x kTile
  for (int idx = threadIdx.x; idx < NB * kTile; idx += 256) {
    const int j = idx % NB, ii = idx / NB;
    su[idx] = (i0 + ii < NB) ? U[((size_t)k * NB + i0 + ii) * NB + j] : cplx<double>{0.0, 0.0};
  }
  __syncthreads();
  if (p >= NL) return;
  const cplx<double>* Ak = A + (size_t)k * NB * NL;
  double re[kTile], im[kTile];
#pragma unroll
  for (int ii = 0; ii < kTile; ++ii) { re[ii] = 0.0; im[ii] = 0.0; }
  for (int j = 0; j < NB; ++j) {
    const cplx<double> a = Ak[(size_t)j * NL + p];
#pragma unroll
    for (int ii = 0; ii < kTile; ++ii) {
      const cplx<double> u = su[ii * NB + j];
      re[ii] += a.re * u.re - a.im * u.im;
      im[ii] += a.re * u.im + a.im * u.re;
    }
  }
#pragma unroll
  for (int ii = 0; ii < kTile; ++ii)
    if (i0 + ii < NB) C[((size_t)k * NB + i0 + ii) * NL + p] = cplx<double>{re[ii], im[ii]};
}

// Gram-Schmidt step of band ib in place (Gram_Schmidt_ompk,
// ARTED/GS/Gram_Schmidt.f90:43-50): v -= sum_{j<ib} zs_j B_j; with_norm ends
// with SN = 1/sqrt(|v|^2 Hxyz).  check_done: not of k points whose done flag is set.
// Grid (nvec, NK).
__global__ void __launch_bounds__(256) k_gs_sub(State S, cplx<double>* __restrict__ zu, int ib, int with_norm,
                                                int check_done) {
  const int k = blockIdx.y, c = blockIdx.x;
  if (check_done && S.done[k]) return;
  cplx<double>* B = zu + (size_t)k * S.NB * S.NL;
  cplx<double>* v = B + (size_t)ib * S.NL;
  const cplx<double>* zs = S.zs + (size_t)k * S.NB;
  const int p = c * 256 + threadIdx.x;
  double a[1] = {0.0};
  if (p < S.NL) {
    cplx<double> e = v[p];
#pragma unroll 8
    for (int j = 0; j < ib; ++j) {
      const cplx<double> b = B[(size_t)j * S.NL + p], z = zs[j];
      e.re -= b.re * z.re - b.im * z.im;
      e.im -= b.re * z.im + b.im * z.re;
    }
    v[p] = e;
    a[0] = e.re * e.re + e.im * e.im;
  }
  if (!with_norm) return;
  double tot[1];
  if (!last_block_sum<1>(a, S, S.nvec, c, tot)) return;
  if (threadIdx.x == 0) S.sc[k * kNS + SN] = 1.0 / sqrt(tot[0] * S.Hxyz);
}

// band ib *= SN.  Grid (nvec, NK).
__global__ void __launch_bounds__(256) k_gs_scale(State S, cplx<double>* __restrict__ zu, int ib, int check_done) {
  const int k = blockIdx.y;
  if (check_done && S.done[k]) return;
  const double f = S.sc[k * kNS + SN];
  cplx<double>* v = zu + ((size_t)k * S.NB + ib) * S.NL;
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p < S.NL) {
    v[p].re *= f;
    v[p].im *= f;
  }
}

// Training sample of the learned preconditioner: the orthogonalised residual
// and the iterate of k = 0, with the band and <x|H|x>.  valid = 0 when the
// band has already left its iterations.
__global__ void __launch_bounds__(256) k_pc_record(State S, const cplx<double>* __restrict__ g,
                                                   const cplx<double>* __restrict__ x, cplx<double>* __restrict__ sg,
                                                   cplx<double>* __restrict__ sx, double* __restrict__ theta,
                                                   int* __restrict__ sib, int* __restrict__ valid, int ib) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < S.NL) {
    sg[i] = g[i];
    sx[i] = x[i];
  }
  if (i == 0) {
    theta[0] = S.sc[XHX];
    sib[0] = ib;
    valid[0] = S.done[0] ? 0 : 1;
  }
}

}  // namespace cg
}  // namespace salmon
