// Host side of the ground-state path: CG_ompk (ARTED/GS/CG.f90:34-139) on
// the resident orbitals with an optional preconditioner, the subspace
// diagonalisation diag_omp (ARTED/GS/diag.f90:95-130), and the sweep loop of
// the ground-state driver (ARTED/control/ground_state.f90:136-140) with a
// frozen potential.  Included by salmon_gpu.hip after its helpers.
#pragma once
#include "cg.hpp"
#include "gsblock.hpp"

using namespace salmon::cg;

// Inference buffers of the learned preconditioner (one residual per k point).
struct PcInfer {
  int NK = 0, NL = 0;
  std::vector<void*> bufs;
  unsigned short *ub = nullptr, *a1b = nullptr, *a2b = nullptr;  // BF16 activations
  float* y = nullptr;
  double *stats = nullptr, *part = nullptr;
};

struct GsState {
  int NK = 0, NB = 0, NL = 0, Nlma = 0, NPI = 0, nchunk = 0, ngroup = 0;
  std::vector<void*> bufs;
  cplx<double>* w[10] = {};  // X HX TX G P PKO HP TP KG T1, NK*NL each
  cplx<double>* ph = nullptr;   // (NK, NPI) phases of the sphere points at the CG's k
  cplx<double>* dps = nullptr;  // (NK, NPI) KB term of each
  double* sc = nullptr;
  int* done = nullptr;
  int* iters = nullptr;
  double* esp_var = nullptr;
  double* part = nullptr;
  unsigned* cnt = nullptr;
  cplx<double>* zs = nullptr;
  cplx<double>* gram = nullptr;
  cplx<double>* minv = nullptr;  // (I + L)^-1 rows of the lower-band triangle
  double* minvr = nullptr;       // (I + Re L)^-1 rows
  double* tw = nullptr;    // DFT twiddles (3*kDftMax complex)
  double* symb = nullptr;  // kinetic symbol per axis (3*kDftMax)
  int pstride = 0;
  GsBlock gsb{};  // panel Gram-Schmidt
  // subspace matrices
  double* dpart = nullptr;
  size_t dpart_n = 0;
  double* dM = nullptr;
  cplx<double>* dU = nullptr;
  int dk = 0;  // k points per subspace pass
  // learned preconditioner: inference buffers, recorded training samples of
  // k = 0 (orthogonalised residual, iterate, band, <x|H|x>) and the targets
  PcInfer inf;
  int smp_cap = 0, smp_n = 0, smp_stride = 1;
  long smp_seen = 0;  // iterations seen while recording
  bool recording = false;
  std::vector<void*> smp_bufs;
  cplx<double>* smp_g = nullptr;
  cplx<double>* smp_x = nullptr;
  double* smp_theta = nullptr;
  int* smp_ib = nullptr;
  int* smp_valid = nullptr;
  std::vector<int> h_ib, h_valid;
  std::vector<double> h_theta;
  cplx<double>* Zc = nullptr;  // (NB, NL) converged bands
  std::vector<double> lam;     // their energies
  // captured launch sequences: a CG call (keyed by its arguments) and a
  // Gram-Schmidt pass (keyed by the orbital array); the first call of a key
  // runs eagerly, later ones capture once and replay
  struct Graph {
    hipGraphExec_t exec = nullptr;
    long key[4] = {-1, -1, -1, -1};
    long warm[4] = {-1, -1, -1, -1};
    unsigned long gen = 0;  // the context's buffer generation of key and warm
  } g_cg, g_gs;
};

static void graph_free(GsState::Graph& g) {
  if (g.exec) (void)hipGraphExecDestroy(g.exec);
  g.exec = nullptr;
  for (int i = 0; i < 4; ++i) g.key[i] = g.warm[i] = -1;
}

static int pc_infer(salmon_ctx* c, GsState* s, salmon_pcnet* net, const cplx<double>* g, cplx<double>* out);

enum { W_X = 0, W_HX, W_TX, W_G, W_P, W_PKO, W_HP, W_TP, W_KG, W_T1 };

static void gs_free(salmon_ctx* c) {
  GsState* s = (GsState*)c->gs;
  if (!s) return;
  for (void* p : s->bufs) (void)hipFree(p);
  (void)hipFree(s->ph);
  (void)hipFree(s->dps);
  for (void* p : s->smp_bufs) (void)hipFree(p);
  for (void* p : s->inf.bufs) (void)hipFree(p);
  graph_free(s->g_cg);
  graph_free(s->g_gs);
  delete s;
  c->gs = nullptr;
}

template <typename X>
static int gs_alloc(salmon_ctx* c, GsState* s, X** p, size_t n) {
  if (n == 0) n = 1;
  hipError_t e = hipMalloc((void**)p, n * sizeof(X));
  if (e != hipSuccess) return fail(c, SALMON_ERR_NOMEM, "ground-state buffers (%zu bytes): %s", n * sizeof(X), hipGetErrorString(e));
  s->bufs.push_back((void*)*p);
  return SALMON_OK;
}

// Finite-difference kinetic symbol of one axis, -1/2 (lap0 + 2 sum_m lap_m
// cos(m 2 pi c/n)), c = 0..n-1, and the DFT twiddles (cos, sin)(2 pi j/n).
static void kinetic_tables(const Grid& g, std::vector<double>& tw, std::vector<double>& symb) {
  tw.assign(2 * 3 * kDftMax, 0.0);
  symb.assign(3 * kDftMax, 0.0);
  const int N[3] = {g.NLx, g.NLy, g.NLz};
  for (int ax = 0; ax < 3; ++ax) {
    const int n = N[ax];
    for (int j = 0; j < n; ++j) {
      const double th = 2.0 * M_PI * j / n;
      tw[2 * (ax * kDftMax + j)] = cos(th);
      tw[2 * (ax * kDftMax + j) + 1] = sin(th);
      double sym = g.lap[ax][0];
      for (int m = 1; m <= 4; ++m) sym += 2.0 * g.lap[ax][m] * cos(m * th);
      symb[ax * kDftMax + j] = -0.5 * sym;
    }
  }
}

// The tables of the sphere points, whose number changes when an atom moves; the
// rest of the state, recorded samples and targets among it, does not depend on them.
static int gs_ensure_points(salmon_ctx* c, GsState* s) {
  if (s->ph && s->NPI == c->kb.NPI) return SALMON_OK;
  (void)hipFree(s->ph);
  (void)hipFree(s->dps);
  s->ph = s->dps = nullptr;
  s->NPI = c->kb.NPI;
  const size_t bytes = sizeof(cplx<double>) * std::max<size_t>(1, (size_t)s->NK * s->NPI);
  if (hipMalloc((void**)&s->dps, bytes) != hipSuccess || hipMalloc((void**)&s->ph, bytes) != hipSuccess) {
    (void)hipFree(s->dps);
    s->ph = s->dps = nullptr;
    return fail(c, SALMON_ERR_NOMEM, "ground-state sphere points (%zu bytes)", bytes);
  }
  return SALMON_OK;
}

static int gs_ensure(salmon_ctx* c) {
  GsState* s = (GsState*)c->gs;
  if (s && s->NK == c->NK && s->NB == c->NB && s->Nlma == c->kb.Nlma) return gs_ensure_points(c, s);
  gs_free(c);
  s = new GsState();
  c->gs = s;
  s->NK = c->NK;
  s->NB = c->NB;
  s->NL = c->g.NL;
  s->Nlma = c->kb.Nlma;
  s->nchunk = (s->NL + kChunk - 1) / kChunk;
  s->ngroup = (s->NB + kJG - 1) / kJG;
  s->pstride = std::max(s->nchunk * s->ngroup * kPartQ, (s->NL + kSubPts - 1) / kSubPts * 5);
  const size_t nv = (size_t)s->NK * s->NL;
  int r;
  for (int i = 0; i < 10; ++i)
    if ((r = gs_alloc(c, s, &s->w[i], nv))) return r;
  if ((r = gs_ensure_points(c, s))) return r;
  if ((r = gs_alloc(c, s, &s->sc, (size_t)s->NK * kNS))) return r;
  if ((r = gs_alloc(c, s, &s->done, (size_t)s->NK))) return r;
  if ((r = gs_alloc(c, s, &s->iters, (size_t)s->NK * s->NB))) return r;
  if ((r = gs_alloc(c, s, &s->esp_var, (size_t)s->NK * s->NB))) return r;
  if ((r = gs_alloc(c, s, &s->part, (size_t)s->NK * s->pstride))) return r;
  if ((r = gs_alloc(c, s, &s->cnt, (size_t)s->NK))) return r;
  if ((r = gs_alloc(c, s, &s->zs, (size_t)s->NK * s->NB))) return r;
  if ((r = gs_alloc(c, s, &s->gram, (size_t)s->NK * s->NB * s->NB))) return r;
  if ((r = gs_alloc(c, s, &s->minv, (size_t)s->NK * s->NB * s->NB))) return r;
  if ((r = gs_alloc(c, s, &s->minvr, (size_t)s->NK * s->NB * s->NB))) return r;
  if ((r = gs_alloc(c, s, &s->tw, (size_t)2 * 3 * kDftMax))) return r;
  if ((r = gs_alloc(c, s, &s->symb, (size_t)3 * kDftMax))) return r;
  GsBlock& q = s->gsb;
  q.NK = s->NK;
  q.NB = s->NB;
  q.NL = s->NL;
  q.Hxyz = c->g.Hxyz;
  q.ntile = (s->NB + kPanel - 1) / kPanel;
  // about 1024 blocks, chunks of at least 1024 points: each 64 bands x 32^3 sweep took 44.4 ms
  // with 1024, 44.5 with 512 and 44.8 with 2048; ten steps of 276 x 20x20x28, reorthonormalised
  // every fifth, 3.30, 3.42 and 3.33
  q.nchunk = std::max(1, std::min(1024 / (s->NK * q.ntile), (s->NL + 1023) / 1024));
  q.chunk = ((s->NL + q.nchunk - 1) / q.nchunk + 63) / 64 * 64;
  q.nchunk = (s->NL + q.chunk - 1) / q.chunk;
  if ((r = gs_alloc(c, s, &q.part, (size_t)s->NK * q.ntile * q.nchunk * 256))) return r;
  if ((r = gs_alloc(c, s, &q.C, (size_t)s->NK * s->NB * kPanel))) return r;
  if ((r = gs_alloc(c, s, &q.W, (size_t)s->NK * s->NB * kPanel))) return r;
  if ((r = gs_alloc(c, s, &q.cnt, (size_t)s->NK * (q.ntile + 1)))) return r;
  if ((r = gs_alloc(c, s, &q.fine, s->NK))) return r;
  HIPCHK(c, hipMemsetAsync(q.cnt, 0, sizeof(unsigned) * s->NK * (q.ntile + 1), c->stream));
  HIPCHK(c, hipMemsetAsync(s->cnt, 0, sizeof(unsigned) * s->NK, c->stream));
  HIPCHK(c, hipMemsetAsync(s->sc, 0, sizeof(double) * s->NK * kNS, c->stream));
  HIPCHK(c, hipMemsetAsync(s->done, 0, sizeof(int) * s->NK, c->stream));
  std::vector<double> tw, symb;
  kinetic_tables(c->g, tw, symb);
  HIPCHK(c, hipMemcpyAsync(s->tw, tw.data(), sizeof(double) * tw.size(), hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipMemcpyAsync(s->symb, symb.data(), sizeof(double) * symb.size(), hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return SALMON_OK;
}

static State gs_view(salmon_ctx* c, GsState* s) {
  State S{};
  S.sc = s->sc;
  S.done = s->done;
  S.iters = s->iters;
  S.esp_var = s->esp_var;
  S.part = s->part;
  S.cnt = s->cnt;
  S.zs = s->zs;
  S.gram = s->gram;
  S.minv = s->minv;
  S.minvr = s->minvr;
  S.occ = c->d_occ;
  S.NK = s->NK;
  S.NB = s->NB;
  S.NL = s->NL;
  S.nchunk = s->nchunk;
  S.nsub = (s->NL + kSubPts - 1) / kSubPts;
  S.nvec = (s->NL + 255) / 256;
  S.pstride = s->pstride;
  S.Hxyz = c->g.Hxyz;
  return S;
}

// K g for the kinetic preconditioner.
static int kinetic_apply(salmon_ctx* c, GsState* s, const State& S, const cplx<double>* g, cplx<double>* out) {
  namespace dft = salmon::dft;
  const Grid& G = c->g;
  const long planes = (long)G.NLx * s->NK;
  const int nz = dft::plane_lines(G.NLz, G.NLy, planes), ny = dft::plane_lines(G.NLy, G.NLz, planes);
  hipLaunchKernelGGL(k_kin_zy, dim3((G.NLz + nz - 1) / nz, G.NLx, s->NK), dim3(256), dft::plane_lds(G.NLz, G.NLy, nz), c->stream, S,
                     g, s->w[W_T1], G, nz, (const double*)s->tw);
  hipLaunchKernelGGL(k_kin_x, dim3(dft::lines_x_blocks(G), s->NK), dim3(256), 0, c->stream, S, s->w[W_T1], G,
                     (const double*)s->tw, (const double*)s->symb);
  hipLaunchKernelGGL(k_kin_yz, dim3((G.NLy + ny - 1) / ny, G.NLx, s->NK), dim3(256), dft::plane_lds(G.NLy, G.NLz, ny), c->stream, S,
                     (const cplx<double>*)s->w[W_T1], out, G, ny, (const double*)s->tw);
  LAUNCHCHK(c);
  return SALMON_OK;
}

// CG_ompk over all bands of all k (FP64 orbitals).  An iteration is a chain of
// launches each too short to hide its start and its reduction's end, so its
// steps share launches where one's results are the next one's operands: nine
// launches without a preconditioner became six (the scalings go with the H
// application and the rotation, the 2x2 sums with the H application, the update
// of the search direction with its orthogonalisation).
static int cg_run(salmon_ctx* c, int ncg, int precond) {
  GsState* s = (GsState*)c->gs;
  State S = gs_view(c, s);
  cplx<double>* zu = (cplx<double>*)c->d_zu;
  cplx<double>** w = s->w;
  const int NK = s->NK, NB = s->NB, NL = s->NL;
  const dim3 gv(S.nvec, NK), blk(256), gsub(S.nsub, NK);
  const size_t bstride = (size_t)NB * NL;
  const bool kinetic = precond == SALMON_PC_KINETIC;
  cplx<double>*const tx = kinetic ? w[W_TX] : nullptr, *const tp = kinetic ? w[W_TP] : nullptr;
  int r;
  if (c->kb.Nlma > 0) {
    hipLaunchKernelGGL(k_phase_table<double>, dim3(((long)NK * c->kb.NPI + 255) / 256), blk, 0, c->stream,
                       (const double*)c->d_kac, NK, 0.0, 0.0, 0.0, c->kb, s->ph);
    LAUNCHCHK(c);
  }
  // H of the vector v; its scaled copy (H_START, H_EFIN) into xo
  auto H = [&](auto role, const cplx<double>* v, cplx<double>* hv, cplx<double>* tv, cplx<double>* xo, size_t xstride,
               int ib, int it) -> int {
    constexpr int R = decltype(role)::value;
    Region reg(c, SALMON_LOG_HPSI);
    if (c->kb.Nlma > 0) {
      hipLaunchKernelGGL(k_cg_kb, dim3(c->kb.NI, NK), blk, 0, c->stream, S, v, c->kb, (const cplx<double>*)s->ph, s->dps,
                         R == H_RR ? 1 : 0);
      LAUNCHCHK(c);
    }
    hipLaunchKernelGGL(k_cg_h<R>, gv, blk, 0, c->stream, S, v, (const double*)c->d_kac, (const double*)c->d_vloc, c->g,
                       c->kb, (const cplx<double>*)s->dps, hv, tv, xo, xstride, (const cplx<double>*)w[W_X], ib, it);
    LAUNCHCHK(c);
    return SALMON_OK;
  };
  auto proj = [&](int ib, Src src, int mode, int check) -> int {
    if (ib == 0) return SALMON_OK;
    hipLaunchKernelGGL(k_cg_proj, dim3(s->nchunk, (ib + kJG - 1) / kJG, NK), blk, 0, c->stream, S,
                       (const cplx<double>*)zu, ib, src, mode, check);
    LAUNCHCHK(c);
    return SALMON_OK;
  };
  auto sub = [&](int ib, Src src, cplx<double>* out, const cplx<double>* other, int role, int it) -> int {
    hipLaunchKernelGGL(k_cg_sub, gsub, dim3(kWide), 0, c->stream, S, (const cplx<double>*)zu, ib, src, out, other,
                       (const cplx<double>*)w[W_X], (const cplx<double>*)w[W_P], role, it, ncg);
    LAUNCHCHK(c);
    return SALMON_OK;
  };
  const Src resid{nullptr, 0, w[W_HX], w[W_X]};
  for (int ib = 0; ib < NB; ++ib) {
    const Src start{zu + (size_t)ib * NL, bstride, nullptr, nullptr};
    // start vector orthogonalised to the lower bands and normalised (CG.f90:67-74)
    if ((r = proj(ib, start, PROJ_START, 0))) return r;
    if ((r = sub(ib, start, w[W_T1], nullptr, SUB_START, 0))) return r;
    if ((r = H(std::integral_constant<int, H_START>(), w[W_T1], w[W_HX], tx, w[W_X], (size_t)NL, ib, 0))) return r;
    for (int it = 1; it <= ncg; ++it) {
      // residual orthogonalised to the lower bands (CG.f90:85-90)
      if ((r = proj(ib, resid, PROJ_VEC, 1))) return r;
      const cplx<double>* dir = w[W_G];
      if ((r = sub(ib, resid, w[W_G], nullptr, precond == SALMON_PC_NONE ? SUB_GRAD : SUB_NONE, it))) return r;
      if (s->recording && s->smp_n < s->smp_cap && NK == 1 && (s->smp_seen++ % s->smp_stride) == 0) {
        const int slot = s->smp_n++;
        hipLaunchKernelGGL(k_pc_record, dim3((NL + 255) / 256), blk, 0, c->stream, S, (const cplx<double>*)w[W_G],
                           (const cplx<double>*)w[W_X], s->smp_g + (size_t)slot * NL, s->smp_x + (size_t)slot * NL,
                           s->smp_theta + slot, s->smp_ib + slot, s->smp_valid + slot, ib);
        LAUNCHCHK(c);
      }
      if (precond != SALMON_PC_NONE) {
        if (precond == SALMON_PC_LEARNED) {
          if ((r = pc_infer(c, s, (salmon_pcnet*)c->pcnet, w[W_G], w[W_KG]))) return r;
        } else {
          if ((r = kinetic_apply(c, s, S, w[W_G], w[W_KG]))) return r;
        }
        const Src kg{w[W_KG], (size_t)NL, nullptr, nullptr};
        if ((r = proj(ib, kg, PROJ_VEC, 1))) return r;
        if ((r = sub(ib, kg, w[W_KG], w[W_G], precond == SALMON_PC_LEARNED ? SUB_LEARN : SUB_PCDIR, it))) return r;
        dir = w[W_KG];
      }
      // search direction, orthogonalised to x and normalised (CG.f90:92-106)
      hipLaunchKernelGGL(k_cg_pko, gv, blk, 0, c->stream, S, dir, w[W_P], (const cplx<double>*)w[W_X], w[W_PKO]);
      LAUNCHCHK(c);
      // its H, the 2x2 Rayleigh-Ritz and the update (CG.f90:107-119)
      if ((r = H(std::integral_constant<int, H_RR>(), w[W_PKO], w[W_HP], tp, nullptr, 0, ib, it))) return r;
      hipLaunchKernelGGL(k_cg_rotate, gv, blk, 0, c->stream, S, w[W_X], w[W_HX], tx, (const cplx<double>*)w[W_PKO],
                         (const cplx<double>*)w[W_HP], (const cplx<double>*)tp);
      LAUNCHCHK(c);
    }
    // store the normalised band and its residual (CG.f90:122-126)
    cplx<double>* band = zu + (size_t)ib * NL;
    if ((r = H(std::integral_constant<int, H_EFIN>(), w[W_X], w[W_HP], nullptr, band, bstride, ib, 0))) return r;
    // row ib of the lower bands' Gram matrix, for the later bands' projections
    if (ib + 1 < NB && (r = proj(ib, Src{band, bstride, nullptr, nullptr}, PROJ_GRAM, 0))) return r;
    hipLaunchKernelGGL(k_cg_resid, gv, blk, 0, c->stream, S, (const cplx<double>*)band, bstride,
                       (const cplx<double>*)w[W_HP], ib);
    LAUNCHCHK(c);
  }
  return SALMON_OK;
}

// Gram_Schmidt_ompk (ARTED/GS/Gram_Schmidt.f90:41-51) on the resident FP64
// orbitals, all k at once and every band over the whole chip: the sequential
// loop's overlaps are taken against the unmodified band and the subtraction
// is repeated once (classical Gram-Schmidt twice, equal to the reference's
// modified form up to rounding), then the band is normalised.
static int gram_schmidt_multi(salmon_ctx* c, cplx<double>* zu, int* skip = nullptr) {
  int r;
  if ((r = gs_ensure(c))) return r;
  GsState* s = (GsState*)c->gs;
  State S = gs_view(c, s);
  const int check = skip ? 1 : 0;
  if (skip) S.done = skip;
  const dim3 gv(S.nvec, s->NK), blk(256);
  for (int ib = 0; ib < s->NB; ++ib) {
    const Src v{zu + (size_t)ib * s->NL, (size_t)s->NB * s->NL, nullptr, nullptr};
    for (int pass = 0; pass < 2 && ib > 0; ++pass) {
      for (int b0 = 0; b0 < ib; b0 += kCgMaxNB) {
        const int nb = std::min(kCgMaxNB, ib - b0);
        State P = S;
        P.zs += b0;
        hipLaunchKernelGGL(k_cg_proj, dim3(s->nchunk, (nb + kJG - 1) / kJG, s->NK), blk, 0, c->stream, P,
                           (const cplx<double>*)zu + (size_t)b0 * s->NL, nb, v, (int)PROJ_PLAIN, check);
        LAUNCHCHK(c);
      }
      hipLaunchKernelGGL(k_gs_sub, gv, blk, 0, c->stream, S, zu, ib, pass == 1 ? 1 : 0, check);
      LAUNCHCHK(c);
    }
    if (ib == 0) {
      hipLaunchKernelGGL(k_gs_sub, gv, blk, 0, c->stream, S, zu, 0, 1, check);
      LAUNCHCHK(c);
    }
    hipLaunchKernelGGL(k_gs_scale, gv, blk, 0, c->stream, S, zu, ib, check);
    LAUNCHCHK(c);
  }
  return SALMON_OK;
}

// Gram_Schmidt_ompk in panels (gsblock.hpp); *done = 0 if a panel of some k point could
// not be orthogonalised so, whose fine flag is then zero (waits for the stream).
static int gram_schmidt_panels(salmon_ctx* c, cplx<double>* zu, int* done) {
  int r;
  if ((r = gs_ensure(c))) return r;
  GsState* s = (GsState*)c->gs;
  GsBlock b = s->gsb;
  b.zu = zu;
  HIPCHK(c, hipMemsetAsync(b.fine, 1, sizeof(int) * b.NK, c->stream));
  for (int j0 = 0; j0 < b.NB; j0 += kPanel) {
    const int np = std::min(kPanel, b.NB - j0);
    for (int round = 0; round < 2; ++round) {
      hipLaunchKernelGGL(k_gsb_overlap, dim3(b.nchunk, (j0 + np + kPanel - 1) / kPanel, b.NK), dim3(256), 0, c->stream, b,
                         j0, np);
      hipLaunchKernelGGL(k_gsb_apply, dim3((b.NL + 63) / 64, b.NK), dim3(256), 0, c->stream, b, j0, np);
      LAUNCHCHK(c);
    }
  }
  std::vector<int> fine(b.NK);
  HIPCHK(c, hipMemcpyAsync(fine.data(), b.fine, sizeof(int) * b.NK, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  *done = std::all_of(fine.begin(), fine.end(), [](int f) { return f != 0; });
  return SALMON_OK;
}

// Runs `enqueue` through the graph cache: eagerly on the first call of a key
// (buffers are allocated there), captured and instantiated on the second,
// replayed afterwards.  A captured graph holds the device pointers of its
// launches, so it is dropped (and the key starts over eagerly) once the
// context has freed or replaced any buffer since (salmon_ctx::gen).  A failed
// capture leaves the key to eager launches.
template <typename F>
static int graph_run(salmon_ctx* c, GsState::Graph& g, const long key[4], F enqueue) {
  if (!c->graphs) return enqueue();
  if (g.gen != c->gen) {
    graph_free(g);
    g.gen = c->gen;
  }
  const bool same = std::equal(key, key + 4, g.key);
  if (g.exec && same) {
    HIPCHK(c, hipGraphLaunch(g.exec, c->stream));
    return SALMON_OK;
  }
  if (!std::equal(key, key + 4, g.warm)) {
    const int r = enqueue();
    // buffers allocated by this eager call belong to the generation a capture will see
    g.gen = c->gen;
    std::copy(key, key + 4, g.warm);
    return r;
  }
  graph_free(g);
  std::copy(key, key + 4, g.warm);
  const unsigned long gen0 = c->gen;
  hipGraph_t graph = nullptr;
  HIPCHK(c, hipStreamBeginCapture(c->stream, hipStreamCaptureModeRelaxed));
  const int r = enqueue();
  const hipError_t e = hipStreamEndCapture(c->stream, &graph);
  if (r) {
    if (graph) (void)hipGraphDestroy(graph);
    return r;
  }
  if (e != hipSuccess || !graph) return fail(c, SALMON_ERR_HIP, "stream capture: %s", hipGetErrorString(e));
  if (c->gen != gen0) {
    // a buffer was replaced while the launches were recorded: run them
    // eagerly instead and capture on a later call
    (void)hipGraphDestroy(graph);
    g.gen = c->gen;
    for (int i = 0; i < 4; ++i) g.warm[i] = -1;
    return enqueue();
  }
  hipGraphExec_t exec = nullptr;
  const hipError_t ei = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  if (ei != hipSuccess) return fail(c, SALMON_ERR_HIP, "graph instantiate: %s", hipGetErrorString(ei));
  g.exec = exec;
  std::copy(key, key + 4, g.key);
  HIPCHK(c, hipGraphLaunch(g.exec, c->stream));
  return SALMON_OK;
}

// ---------------------------------------------------------------------------
// Eigenpairs of a Hermitian matrix (row-major n x n) by cyclic Jacobi
// rotations; eigenvalues ascending, eigenvectors as the columns of V.
// ---------------------------------------------------------------------------
struct zc64 {
  double re, im;
};

static void jacobi_herm(int n, std::vector<zc64>& A, std::vector<double>& w, std::vector<zc64>& V) {
  auto a = [&](int i, int j) -> zc64& { return A[(size_t)i * n + j]; };
  V.assign((size_t)n * n, zc64{0, 0});
  for (int i = 0; i < n; ++i) V[(size_t)i * n + i].re = 1.0;
  double fro = 0.0;
  for (int i = 0; i < n; ++i)
    for (int j = 0; j < n; ++j) fro += a(i, j).re * a(i, j).re + a(i, j).im * a(i, j).im;
  for (int sweep = 0; sweep < 100; ++sweep) {
    double off = 0.0;
    for (int i = 0; i < n; ++i)
      for (int j = i + 1; j < n; ++j) off += a(i, j).re * a(i, j).re + a(i, j).im * a(i, j).im;
    if (off <= 1e-30 * fro || off == 0.0) break;
    for (int p = 0; p < n; ++p) {
      for (int q = p + 1; q < n; ++q) {
        const zc64 apq = a(p, q);
        const double gabs = std::hypot(apq.re, apq.im);
        if (gabs == 0.0) continue;
        const zc64 e{apq.re / gabs, apq.im / gabs};  // a_pq = g e
        const double tau = (a(q, q).re - a(p, p).re) / (2.0 * gabs);
        const double t = (tau >= 0 ? 1.0 : -1.0) / (std::fabs(tau) + std::sqrt(1.0 + tau * tau));
        const double cs = 1.0 / std::sqrt(1.0 + t * t), sn = t * cs;
        // U: U_pp = c, U_pq = s e, U_qp = -s conj(e), U_qq = c;  A <- U^H A U, V <- V U
        for (int k = 0; k < n; ++k) {  // columns: A U
          const zc64 akp = a(k, p), akq = a(k, q);
          // akp' = c akp - s conj(e) akq ; akq' = s e akp + c akq
          a(k, p) = zc64{cs * akp.re - sn * (e.re * akq.re + e.im * akq.im), cs * akp.im - sn * (e.re * akq.im - e.im * akq.re)};
          a(k, q) = zc64{sn * (e.re * akp.re - e.im * akp.im) + cs * akq.re, sn * (e.re * akp.im + e.im * akp.re) + cs * akq.im};
          const zc64 vkp = V[(size_t)k * n + p], vkq = V[(size_t)k * n + q];
          V[(size_t)k * n + p] = zc64{cs * vkp.re - sn * (e.re * vkq.re + e.im * vkq.im), cs * vkp.im - sn * (e.re * vkq.im - e.im * vkq.re)};
          V[(size_t)k * n + q] = zc64{sn * (e.re * vkp.re - e.im * vkp.im) + cs * vkq.re, sn * (e.re * vkp.im + e.im * vkp.re) + cs * vkq.im};
        }
        for (int k = 0; k < n; ++k) {  // rows: U^H B
          const zc64 bpk = a(p, k), bqk = a(q, k);
          // bpk' = c bpk - s e bqk ; bqk' = s conj(e) bpk + c bqk
          a(p, k) = zc64{cs * bpk.re - sn * (e.re * bqk.re - e.im * bqk.im), cs * bpk.im - sn * (e.re * bqk.im + e.im * bqk.re)};
          a(q, k) = zc64{sn * (e.re * bpk.re + e.im * bpk.im) + cs * bqk.re, sn * (e.re * bpk.im - e.im * bpk.re) + cs * bqk.im};
        }
        a(p, q) = zc64{0, 0};
        a(q, p) = zc64{0, 0};
        a(p, p).im = 0.0;
        a(q, q).im = 0.0;
      }
    }
  }
  std::vector<int> ord(n);
  for (int i = 0; i < n; ++i) ord[i] = i;
  std::stable_sort(ord.begin(), ord.end(), [&](int x, int y) { return a(x, x).re < a(y, y).re; });
  std::vector<zc64> W((size_t)n * n);
  w.resize(n);
  for (int i = 0; i < n; ++i) {
    w[i] = a(ord[i], ord[i]).re;
    for (int k = 0; k < n; ++k) W[(size_t)k * n + i] = V[(size_t)k * n + ord[i]];
  }
  V.swap(W);
}

// diag_omp: za = <psi_i|H psi_j> Hxyz, eigenvectors U, zu <- zu U, esp = eigenvalues.
static int subspace_diag(salmon_ctx* c, double* esp) {
  GsState* s = (GsState*)c->gs;
  const int NK = c->NK, NB = c->NB, NL = c->g.NL;
  int r;
  if ((r = ensure_work(c))) return r;
  if (c->chunk < NB) return fail(c, SALMON_ERR_UNSUPPORTED, "subspace diagonalisation needs %d orbitals of work space", NB);
  const int nslice = std::max(1, std::min(32, NL / 1024));
  const int pts = ((NL + nslice - 1) / nslice + kSlicePts - 1) / kSlicePts * kSlicePts;
  const size_t per_k = (size_t)nslice * NB * NB * 2;
  int dk = std::max(1, std::min({NK, c->chunk / NB, (int)std::max<size_t>(1, ((size_t)32 << 20) / (per_k * 8))}));
  if (!s->dpart || s->dk != dk) {
    if ((r = gs_alloc(c, s, &s->dpart, per_k * dk))) return r;
    if ((r = gs_alloc(c, s, &s->dM, (size_t)NK * NB * NB * 2))) return r;
    if ((r = gs_alloc(c, s, &s->dU, (size_t)NK * NB * NB))) return r;
    s->dk = dk;
  }
  cplx<double>* zu = (cplx<double>*)c->d_zu;
  cplx<double>* hb = (cplx<double>*)c->d_work[0];
  const int ntile = (NB + kTile - 1) / kTile;
  for (int k0 = 0; k0 < NK; k0 += dk) {
    const int kn = std::min(dk, NK - k0);
    cplx<double>* zk = zu + (size_t)k0 * NB * NL;
    if ((r = apply_h<double>(c, zk, hb, nullptr, k0 * NB, kn * NB, NB, NK, c->d_kac, 0, 0, 0))) return r;
    hipLaunchKernelGGL(k_sub_matrix, dim3(ntile * ntile, nslice, kn), dim3(256), 0, c->stream,
                       (const cplx<double>*)zk, (const cplx<double>*)hb, NB, NL, pts, s->dpart);
    LAUNCHCHK(c);
    hipLaunchKernelGGL(k_sub_matrix_sum, dim3((NB * NB * 2 + 255) / 256, kn), dim3(256), 0, c->stream,
                       (const double*)s->dpart, NB, nslice, c->g.Hxyz, s->dM + (size_t)k0 * NB * NB * 2);
    LAUNCHCHK(c);
  }
  std::vector<double> M((size_t)NK * NB * NB * 2);
  HIPCHK(c, hipMemcpyAsync(M.data(), s->dM, sizeof(double) * M.size(), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  std::vector<zc64> Uall((size_t)NK * NB * NB);
  for (int k = 0; k < NK; ++k) {
    const double* m = &M[(size_t)k * NB * NB * 2];
    // za(ib2,ib1) = <ib2|H|ib1> for ib2 > ib1, za(ib1,ib2) its conjugate,
    // za(ib1,ib1) = Re<ib1|H|ib1> (diag.f90:111-117)
    std::vector<zc64> A((size_t)NB * NB);
    for (int i = 0; i < NB; ++i) {
      A[(size_t)i * NB + i] = zc64{m[2 * ((size_t)i * NB + i)], 0.0};
      for (int j = 0; j < i; ++j) {
        const zc64 v{m[2 * ((size_t)i * NB + j)], m[2 * ((size_t)i * NB + j) + 1]};
        A[(size_t)i * NB + j] = v;
        A[(size_t)j * NB + i] = zc64{v.re, -v.im};
      }
    }
    std::vector<double> w;
    std::vector<zc64> V;
    jacobi_herm(NB, A, w, V);
    for (int i = 0; i < NB; ++i) {
      if (esp) esp[(size_t)k * NB + i] = w[i];
      for (int j = 0; j < NB; ++j) Uall[((size_t)k * NB + i) * NB + j] = V[(size_t)j * NB + i];  // column i
    }
  }
  HIPCHK(c, hipMemcpyAsync(s->dU, Uall.data(), sizeof(zc64) * Uall.size(), hipMemcpyHostToDevice, c->stream));
  // zu(:, i) = sum_j zu(:, j) U(j, i)  (diag.f90:120-127)
  for (int k0 = 0; k0 < NK; k0 += dk) {
    const int kn = std::min(dk, NK - k0);
    cplx<double>* zk = zu + (size_t)k0 * NB * NL;
    hipLaunchKernelGGL(k_rotate_bands, dim3((NL + 255) / 256, ntile, kn), dim3(256), sizeof(cplx<double>) * NB * kTile,
                       c->stream, (const cplx<double>*)zk, (const cplx<double>*)(s->dU + (size_t)k0 * NB * NB), hb, NB, NL);
    LAUNCHCHK(c);
    HIPCHK(c, hipMemcpyAsync(zk, hb, sizeof(cplx<double>) * (size_t)kn * NB * NL, hipMemcpyDeviceToDevice, c->stream));
  }
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return SALMON_OK;
}
