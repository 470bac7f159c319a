// Host side of the batched step: a batch references set-up contexts (their
// orbitals, potentials, tables and k points stay where the contexts put them),
// owns per-system work buffers, tunes the stencil's z blocking per grid shape
// and runs the time loop as replays of one captured step.
#pragma once
#include <array>

#include <algorithm>

#include "batch_sweep.hpp"
#include "resident.hpp"

using namespace salmon::batch;

struct salmon_batch {
  int precision = SALMON_FP64;
  hipStream_t stream = nullptr;
  std::string err;
  std::vector<salmon_ctx*> ctx;
  std::vector<void*> bufs;        // work buffers (rebuilt by prepare)
  void* d_sys = nullptr;          // Sys<T>[n]
  std::vector<int> zb;            // chosen z blocking per system
  std::vector<long> first[kPhases + 1];
  unsigned short* d_owner[kPhases] = {};  // block -> system tables (in bufs)
  long zcls[4][2] = {};                   // stencil blocks of the z-blocking classes 1, 2, 4, 8: (first, count)
  bool ready = false, tuned = false;
  int* d_step = nullptr;
  double* d_ac = nullptr;
  double* d_res = nullptr;
  size_t cap_steps = 0;
  size_t cap_ac = 0;              // doubles in d_ac
  long max_ph = 0;                // largest NK * NPI over the systems
  // persistent sweep (one launch per step) or one launch per phase
  int kernel_req = SALMON_BATCH_AUTO;
  bool sweep = false;
  int2* d_items = nullptr;        // (system, first orbital), costliest first (in bufs)
  int nitems = 0;
  int* d_next = nullptr;          // work counter of the sweep launch; arrivals of the sums' blocks
  // batches of systems whose orbitals fit in LDS (resident.hpp): one launch per
  // workgroup shape (device memory in bufs)
  struct ResClass {
    int px = 0, waves = 0;
    size_t lds = 0;
    const int2* items = nullptr;  // (system, orbital)
    int nitems = 0;
  };
  std::vector<ResClass> res;
  const ResTab* d_restab = nullptr;
  bool resident = false;
  bool resident_ok = true;        // not asked for the sweep itself
  unsigned sweep_grid = 0;
  size_t sweep_lds = 0;
  // one Taylor step at caller-given k points (batch_taylor): descriptors whose
  // kac0 is the given table, a zero A(t) table and a zero step counter (in bufs)
  void* d_sys_k = nullptr;
  const double* const* sys_k_base = nullptr;
  double* d_zero_ac = nullptr;
  int* d_zero_step = nullptr;
  hipGraphExec_t exec = nullptr;
  double graph_dt = 0.0;
  long graph_stride = 0;          // the A(t) table stride the graph was captured with
};

static int bfail(salmon_batch* b, int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  b->err = buf;
  return code;
}

#define BHIP(b, x)                                                                                   \
  do {                                                                                               \
    hipError_t e_ = (x);                                                                             \
    if (e_ != hipSuccess) return bfail((b), SALMON_ERR_HIP, "%s: %s", #x, hipGetErrorString(e_));    \
  } while (0)

static void batch_release(salmon_batch* b) {
  if (b->exec) (void)hipGraphExecDestroy(b->exec);
  b->exec = nullptr;
  for (void* p : b->bufs) (void)hipFree(p);
  b->bufs.clear();
  b->d_sys = nullptr;
  b->d_sys_k = nullptr;
  b->sys_k_base = nullptr;
  b->d_zero_ac = nullptr;
  b->d_zero_step = nullptr;
  for (int ph = 0; ph < kPhases; ++ph) b->d_owner[ph] = nullptr;
  b->d_items = nullptr;
  b->nitems = 0;
  b->res.clear();
  b->d_restab = nullptr;
  b->resident = false;
  b->sweep = false;
  b->ready = false;
}

// Column length (points along z per thread) and team size (waves) of the
// persistent sweep for one grid: the candidate that leaves the fewest team
// threads without a column, the longer column on a tie; {0, 0} if no
// candidate fits a workgroup or the grid is too small for single periodic wraps.
template <typename T>
static std::array<int, 2> sweep_shape(const Grid& g) {
  constexpr int zbmax = sizeof(T) == 4 ? 4 : 2;
  std::array<int, 2> best{0, 0};
  if (g.NLx < 8 || g.NLy < 8 || g.NLz < 8) return best;
  const int P = g.NLy * g.NLz;
  double bu = -1.0;
  for (int zb = 1; zb <= zbmax; ++zb) {
    if (g.NLz % zb) continue;
    const int ncol = P / zb;
    int tw = 1;
    while (tw < sweep_waves<T>() && tw * kWave < ncol) tw *= 2;
    if (tw * kWave < ncol) continue;
    const double u = (double)ncol / (tw * kWave);
    if (u > bu + 1e-12 || (u > bu - 1e-12 && zb > best[0])) {
      bu = u;
      best = {zb, tw};
    }
  }
  return best;
}

// The resident kernel's plan: taken where it covers every system of the batch
// (a grid of its shapes whose orbital, with the sphere points' tables, fits in
// LDS, up to kResLpa projectors per atom, images within two cells) and the
// orbitals are at most kResRounds per compute unit) and is not expected to be
// slower than the sweep by more than its fewer launches give back (resident_pays).
// Beside systems that need the sweep the sweep takes all: its work queue fills the
// chip across systems.  Builds the tables, work lists and rows; b->resident stays
// false if the plan does not apply.
constexpr int kResSteps = 32;  // steps per launch (rows kept per orbital)
constexpr long kResRounds = 4;
constexpr size_t kSweepMaxLds = 65536;

// LDS of the sweep for one system of the given column length and team size
template <typename T>
static size_t sweep_lds_bytes(const Sys<T>& y, const std::array<int, 2>& sh) {
  const int teams = sweep_waves<T>() / sh[1];
  const int zb = sh[0], cs = zb % 2 == 0 ? zb + 1 : zb;  // col_stride<zb>()
  const size_t PS = ((size_t)y.g.NLy * y.g.NLz / zb + 1) * cs;  // plane_slots<zb>(P)
  return (size_t)kSweepHead + (size_t)teams * (2 * PS + y.kb.Nlma) * sizeof(cplx<T>);
}

// Time of one H application of all orbitals in the resident kernel against the
// sweep's.  The resident kernel runs one workgroup per compute unit, so its time is
// its orbitals' times the rounds; the sweep's is a chain of planes that 4 to 8
// orbitals per compute unit run at nearly the time of one.  Fits (us) to 380
// measured pairs (21 grids of 8x8x8 to 18x16x16, 512 to 1024 orbitals, 1 and 6 atoms,
// both precisions), each within 16 % and 4 to 5 % on average: the resident kernel by
// its x points per thread and atoms per wave, the sweep by planes, column length,
// team size and passes over the sphere points, and by how full the chip is.  The
// lines, 1.1 and in complex64 1.25, are where runs of ten steps (which the resident
// kernel needs fewer launches for) took as long either way; with several shapes, a
// launch after another, 0.9.  Without the comparison 14^3 x 1024 orbitals took 194 us a hamiltonian call
// in FP64 where the sweep takes 144, 31x8x9 x 1024 193 and 138; 12^3 x 1024 104
// and 119.
template <typename T>
static bool resident_pays(const salmon_batch* b, const std::vector<Sys<T>>& S, int ncu) {
  constexpr bool f64 = sizeof(T) == 8;
  const double base[7] = {0, f64 ? 2.2 : 2.0, f64 ? 2.9 : 2.6, f64 ? 4.6 : 3.6, f64 ? 6.6 : 4.5, 0, f64 ? 10.8 : 5.9};
  struct Class {
    int px, waves;
    long n;
    double t;
  };
  std::vector<Class> cls;  // a launch each
  long items = 0;
  for (const auto& y : S) {
    const auto sh = sweep_shape<T>(y.g);
    if (sweep_lds_bytes(y, sh) > kSweepMaxLds) return true;  // there is no sweep
    items += (y.NKB + sweep_waves<T>() / sh[1] - 1) / (sweep_waves<T>() / sh[1]);
    const int px = res_px(y.g), waves = res_waves(y.g, px);
    const double t = base[px] + (f64 ? 2.6 : 2.2) * y.kb.NI / waves;
    size_t c = 0;
    while (c < cls.size() && (cls[c].px != px || cls[c].waves != waves)) ++c;
    if (c == cls.size()) cls.push_back({px, waves, 0, 0.0});
    cls[c].n += y.NKB;
    cls[c].t = std::max(cls[c].t, t);
  }
  double res = 0;
  for (const auto& c : cls) res += c.t * ((c.n + ncu - 1) / ncu);
  // the sweep: eight waves per compute unit
  const long slots = (long)ncu * 8 / sweep_waves<T>(), full = items / slots, rest = items % slots;
  double mean = 0, most = 0;  // an item on a full chip; the longest in the last round
  for (size_t i = 0; i < S.size(); ++i) {
    const auto sh = sweep_shape<T>(S[i].g);
    const std::vector<int>& start = b->ctx[i]->kb_host.start;
    long passes = 0;
    for (int a = 0; a < S[i].kb.NI; ++a) passes += (start[a + 1] - start[a] + kWave * sh[1] - 1) / (kWave * sh[1]);
    const double team = std::log2((double)sh[1]);
    const double chain = f64 ? (S[i].g.NLx + 2) * (0.62 * sh[0] + 0.1 * team)
                             : (S[i].g.NLx + 4) * (0.12 + 0.23 * sh[0] + 0.06 * team);
    const double kb = f64 ? 2.4 * passes - 2.0 : 2.3 * passes - 2.5;
    const int teams = sweep_waves<T>() / sh[1];
    mean += (chain * (f64 ? 1.45 : 1.64) + kb) * ((S[i].NKB + teams - 1) / teams) / items;
    most = std::max(most, chain * (1.0 + (f64 ? 0.45 : 0.64) * rest / slots) + kb);
  }
  return res <= (cls.size() > 1 ? 0.9 : f64 ? 1.1 : 1.25) * (full * mean + (rest ? most : 0.0));
}

template <typename T>
static int resident_plan(salmon_batch* b, std::vector<Sys<T>>& S) {
  int dev = 0, ncu = 0;
  BHIP(b, hipGetDevice(&dev));
  BHIP(b, hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
  long orbitals = 0;
  for (const auto& y : S) {
    orbitals += y.NKB;
    const Grid& g = y.g;
    if (!res_px(g) || res_lds<T>(g, y.kb.NPI, y.kb.NI) > kResMaxLds || y.kb.max_lpa > kResLpa || y.kb.NPI >= 0xffff ||
        std::max({g.NLx, g.NLy, g.NLz}) > 200)
      return SALMON_OK;
  }
  if (orbitals > kResRounds * ncu || !resident_pays<T>(b, S, ncu)) return SALMON_OK;
  // all tables and work lists in one device block: offsets first, pointers after its allocation
  std::vector<unsigned char> blob;
  auto put = [&](const void* src, size_t bytes) {
    const size_t at = blob.size();
    blob.resize((at + bytes + 15) / 16 * 16);
    if (bytes) std::memcpy(blob.data() + at, src, bytes);
    return at;
  };
  std::vector<std::array<size_t, 6>> at(S.size());
  std::vector<int> nov(S.size());
  std::vector<std::vector<int2>> items;
  std::vector<salmon_batch::ResClass> res;
  size_t rows = 0;
  for (size_t i = 0; i < S.size(); ++i) {
    const Grid& g = S[i].g;
    const KBTables& kb = S[i].kb;
    const auto& h = b->ctx[i]->kb_host;
    std::vector<int> code(kb.NPI), prim(g.NL, kb.NPI), ovs(1, 0), ovj;
    std::vector<double> uvp((size_t)kb.NPI * kResLpa, 0.0), sgp((size_t)kb.NI * kResLpa, 0.0);
    for (int a = 0; a < kb.NI; ++a)
      for (int l = h.lma[a]; l < h.lma[a + 1]; ++l) {
        sgp[(size_t)a * kResLpa + l - h.lma[a]] = h.sign[l];
        for (int jp = h.start[a]; jp < h.start[a + 1]; ++jp)
          uvp[(size_t)jp * kResLpa + l - h.lma[a]] = h.uv[(size_t)l * kb.Nps + jp - h.start[a]];
      }
    const int N[3] = {g.NLx, g.NLy, g.NLz};
    const double H[3] = {g.Hx, g.Hy, g.Hz}, L[3] = {g.aLx, g.aLy, g.aLz};
    std::vector<int> more(kb.NPI, -1), last(g.NL, -1);  // sphere points of a grid point: prim, then chained in order
    for (int jp = 0; jp < kb.NPI; ++jp) {
      const int p = h.pidx[jp], l[3] = {p / (g.NLy * g.NLz), (p / g.NLz) % g.NLy, p % g.NLz};
      if (last[p] < 0) prim[p] = jp;
      else more[last[p]] = jp;
      last[p] = jp;
      code[jp] = 0;
      for (int d = 0; d < 3; ++d) {
        const int img = (int)std::lround((l[d] * H[d] - h.pos[3 * (size_t)jp + d]) / L[d]);  // pos = l H - img L
        if (img < -2 || img > 2) return SALMON_OK;
        code[jp] |= ((img + 2) * N[d] + l[d]) << (10 * d);
      }
    }
    for (int p = 0; p < g.NL; ++p) {
      if (prim[p] == kb.NPI || more[prim[p]] < 0) continue;
      for (int jp = prim[p]; jp >= 0; jp = more[jp]) ovj.push_back(jp);
      ovs.push_back((int)ovj.size());
    }
    nov[i] = (int)ovs.size() - 1;
    at[i] = {put(prim.data(), sizeof(int) * prim.size()), put(code.data(), sizeof(int) * code.size()),
             put(uvp.data(), sizeof(double) * uvp.size()), put(sgp.data(), sizeof(double) * sgp.size()),
             put(ovs.data(), sizeof(int) * ovs.size()), put(ovj.data(), sizeof(int) * ovj.size())};
    rows += (size_t)8 * kResSteps * S[i].NKB;
    const int px = res_px(g), waves = res_waves(g, px);
    size_t c = 0;
    while (c < res.size() && (res[c].px != px || res[c].waves != waves)) ++c;
    if (c == res.size()) {
      res.emplace_back();
      res[c].px = px;
      res[c].waves = waves;
      items.emplace_back();
    }
    res[c].lds = std::max(res[c].lds, res_lds<T>(g, kb.NPI, kb.NI));
    for (int o = 0; o < S[i].NKB; ++o) items[c].push_back(int2{(int)i, o});
  }
  std::vector<size_t> at_items(res.size());
  for (size_t c = 0; c < res.size(); ++c) at_items[c] = put(items[c].data(), sizeof(int2) * items[c].size());
  std::vector<ResTab> tabs(S.size());
  const size_t at_tabs = put(tabs.data(), sizeof(ResTab) * tabs.size());
  unsigned char* d = nullptr;
  double* d_rows = nullptr;
  if (hipMalloc((void**)&d, blob.size()) != hipSuccess) return bfail(b, SALMON_ERR_NOMEM, "resident tables");
  b->bufs.push_back(d);
  if (hipMalloc((void**)&d_rows, sizeof(double) * rows) != hipSuccess)
    return bfail(b, SALMON_ERR_NOMEM, "resident rows");
  b->bufs.push_back(d_rows);
  for (size_t i = 0; i < S.size(); ++i) {
    tabs[i] = ResTab{(const int*)(d + at[i][0]), (const int*)(d + at[i][1]), (const double*)(d + at[i][2]),
                     (const double*)(d + at[i][3]), (const int*)(d + at[i][4]), (const int*)(d + at[i][5]), nov[i], {}, {}};
    for (int a = 0; a < 3; ++a)
      for (int m = 0; m < 4; ++m) {
        tabs[i].cc[a][m] = -0.5 * S[i].g.lap[a][m + 1];
        tabs[i].dc[a][m] = S[i].g.nab[a][m + 1];
      }
    S[i].rrows = d_rows;
    d_rows += (size_t)8 * kResSteps * S[i].NKB;
  }
  std::memcpy(blob.data() + at_tabs, tabs.data(), sizeof(ResTab) * tabs.size());
  BHIP(b, hipMemcpy(d, blob.data(), blob.size(), hipMemcpyHostToDevice));
  for (size_t c = 0; c < res.size(); ++c) {
    res[c].nitems = (int)items[c].size();
    res[c].items = (const int2*)(d + at_items[c]);
  }
  b->d_restab = (const ResTab*)(d + at_tabs);
  b->res = res;
  b->resident = true;
  return SALMON_OK;
}

template <typename T, int PX>
static int resident_launch_px(salmon_batch* b, const salmon_batch::ResClass& c, const Sys<T>* S, const ResArgs& a) {
  // set once per kernel instantiation (a thread-safe static initialisation)
  static const hipError_t attr = hipFuncSetAttribute((const void*)k_b_resident<T, PX>,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)kResMaxLds);
  BHIP(b, attr);
  hipLaunchKernelGGL((k_b_resident<T, PX>), dim3(c.nitems), dim3(c.waves * kWave), c.lds, b->stream, S,
                     b->d_restab, c.items, a);
  return SALMON_OK;
}

// Steps n0 .. n0 + a.nsteps - 1 (at most kResSteps) of a resident batch, and with
// a.obs their sums into res.
template <typename T>
static int resident_launch(salmon_batch* b, const Sys<T>* S, const ResArgs& a, double* res) {
  int r = SALMON_OK;
  for (const auto& c : b->res) {
    switch (c.px) {
      case 1: r = resident_launch_px<T, 1>(b, c, S, a); break;
      case 2: r = resident_launch_px<T, 2>(b, c, S, a); break;
      case 3: r = resident_launch_px<T, 3>(b, c, S, a); break;
      case 4: r = resident_launch_px<T, 4>(b, c, S, a); break;
      default: r = resident_launch_px<T, 6>(b, c, S, a); break;
    }
    if (r) return r;
  }
  if (a.obs)
    hipLaunchKernelGGL(k_b_resident_sum<T>, dim3((unsigned)b->ctx.size(), a.nsteps), dim3(256), 0, b->stream, S, a.n0, res);
  BHIP(b, hipGetLastError());
  return SALMON_OK;
}

// The persistent sweep's work list, LDS size and grid; b->sweep stays false
// (one launch per phase) if the phase kernel is asked for or, under
// SALMON_BATCH_AUTO, a system does not fit the sweep.
template <typename T>
static int sweep_plan(salmon_batch* b, std::vector<Sys<T>>& S) {
  b->sweep = false;
  if (b->kernel_req == SALMON_BATCH_PHASES) return SALMON_OK;
  const bool must = b->kernel_req == SALMON_BATCH_SWEEP;
  std::vector<std::array<long, 3>> items;  // (cost, system, first orbital)
  size_t lds = 0;
  for (size_t i = 0; i < S.size(); ++i) {
    S[i].kb_order = S[i].kb_cstart = nullptr;
    S[i].ncolor = 0;
  }
  for (size_t i = 0; i < S.size(); ++i) {
    const auto sh = sweep_shape<T>(S[i].g);
    if (!sh[0]) {
      if (must) return bfail(b, SALMON_ERR_ARG, "system %zu (%dx%dx%d) does not fit the persistent sweep", i,
                             S[i].g.NLx, S[i].g.NLy, S[i].g.NLz);
      return SALMON_OK;
    }
    S[i].sw_zb = sh[0];
    S[i].sw_tw = sh[1];
    const int teams = sweep_waves<T>() / sh[1];
    lds = std::max(lds, sweep_lds_bytes(S[i], sh));
    for (int o = 0; o < S[i].NKB; o += teams)
      items.push_back({(long)S[i].g.NL * std::min(teams, S[i].NKB - o), (long)i, (long)o});
  }
  // colours of the atoms of every system: greedy, an atom takes the first
  // colour none of whose atoms shares a grid point with it
  for (size_t i = 0; i < S.size(); ++i) {
    const KBTables& kb = S[i].kb;
    if (kb.NI <= 0 || kb.Nlma <= 0) continue;
    const std::vector<int>&ast = b->ctx[i]->kb_host.start, &pidx = b->ctx[i]->kb_host.pidx;
    std::vector<std::vector<char>> used;
    std::vector<int> colour(kb.NI);
    for (int a = 0; a < kb.NI; ++a) {
      int c = 0;
      for (;; ++c) {
        if (c == (int)used.size()) used.emplace_back(S[i].g.NL, 0);
        bool clash = false;
        for (int jp = ast[a]; jp < ast[a + 1] && !clash; ++jp) clash = used[c][pidx[jp]] != 0;
        if (!clash) break;
      }
      for (int jp = ast[a]; jp < ast[a + 1]; ++jp) used[c][pidx[jp]] = 1;
      colour[a] = c;
    }
    const int nc = (int)used.size();
    std::vector<int> tab;  // kb_order (NI), then kb_cstart (nc + 1)
    std::vector<int> cst(nc + 1, 0);
    for (int c = 0; c < nc; ++c) {
      cst[c] = (int)tab.size();
      for (int a = 0; a < kb.NI; ++a)
        if (colour[a] == c) tab.push_back(a);
    }
    cst[nc] = (int)tab.size();
    tab.insert(tab.end(), cst.begin(), cst.end());
    int* d = nullptr;
    if (hipMalloc((void**)&d, sizeof(int) * tab.size()) != hipSuccess)
      return bfail(b, SALMON_ERR_NOMEM, "batch atom colours");
    b->bufs.push_back(d);
    BHIP(b, hipMemcpy(d, tab.data(), sizeof(int) * tab.size(), hipMemcpyHostToDevice));
    S[i].kb_order = d;
    S[i].kb_cstart = d + kb.NI;
    S[i].ncolor = nc;
  }
  if (lds > kSweepMaxLds || items.empty()) {
    if (must) return bfail(b, SALMON_ERR_ARG, "the persistent sweep needs %zu bytes of LDS", lds);
    return SALMON_OK;
  }
  std::stable_sort(items.begin(), items.end(), [](const std::array<long, 3>& a, const std::array<long, 3>& c) {
    return a[0] > c[0];
  });
  std::vector<int2> it(items.size());
  for (size_t k = 0; k < items.size(); ++k) it[k] = int2{(int)items[k][1], (int)items[k][2]};
  if (hipMalloc((void**)&b->d_items, sizeof(int2) * it.size()) != hipSuccess)
    return bfail(b, SALMON_ERR_NOMEM, "batch work list");
  b->bufs.push_back(b->d_items);
  BHIP(b, hipMemcpy(b->d_items, it.data(), sizeof(int2) * it.size(), hipMemcpyHostToDevice));
  int dev = 0, ncu = 0, per = 0;
  BHIP(b, hipGetDevice(&dev));
  BHIP(b, hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
  const void* kern = nullptr;
  if constexpr (sizeof(T) == 4)
    kern = (const void*)k_b_sweep<T, 4>;
  else
    kern = (const void*)k_b_sweep<T, 2>;
  BHIP(b, hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kern, sweep_waves<T>() * kWave, lds));
  if (per < 1) {
    if (must) return bfail(b, SALMON_ERR_ARG, "the persistent sweep does not fit a compute unit");
    return SALMON_OK;
  }
  b->nitems = (int)it.size();
  b->sweep_lds = lds;
  b->sweep_grid = (unsigned)std::min<long>((long)ncu * per, (long)it.size());
  b->sweep = true;
  return SALMON_OK;
}

template <typename T>
static int batch_build(salmon_batch* b) {
  const int n = (int)b->ctx.size();
  std::vector<Sys<T>> S(n);
  b->max_ph = 0;
  bool sweeps = b->kernel_req != SALMON_BATCH_PHASES && b->resident_ok;
  for (int i = 0; i < n; ++i) {
    salmon_ctx* c = b->ctx[i];
    Sys<T>& y = S[i];
    sweeps = sweeps && sweep_shape<T>(c->g)[0] > 0;
    y.g = c->g;
    y.kb = c->kb;
    y.zu = (cplx<T>*)c->d_zu;
    y.vloc = vloc_ptr<T>(c);
    y.vloc64 = c->d_vloc;
    y.kac0 = c->d_kac0;
    y.occ = c->d_occ;
    y.NK = c->NK;
    y.NB = c->NB;
    y.NKB = c->NKB;
    y.zb = b->zb[i];
    y.sw_zb = y.sw_tw = 0;
    y.rrows = nullptr;
  }
  int r;
  if (sweeps && (r = resident_plan<T>(b, S))) return r;
  long acc[kPhases] = {0, 0, 0, 0, 0};
  for (int i = 0; i < n && !b->resident; ++i) {
    salmon_ctx* c = b->ctx[i];
    Sys<T>& y = S[i];
    const size_t nv = (size_t)c->NKB * c->g.NL;
    for (int t = 0; t < 4; ++t) {
      if (hipMalloc((void**)&y.h[t], nv * sizeof(cplx<T>)) != hipSuccess)
        return bfail(b, SALMON_ERR_NOMEM, "batch work buffers (system %d)", i);
      b->bufs.push_back(y.h[t]);
    }
    if (hipMalloc((void**)&y.uv, (size_t)c->NKB * std::max(1, c->kb.Nlma) * sizeof(cplx<T>)) != hipSuccess ||
        hipMalloc((void**)&y.ph, (size_t)c->NK * std::max(1, c->kb.NPI) * sizeof(cplx<T>)) != hipSuccess ||
        hipMalloc((void**)&y.phn, (size_t)c->NK * std::max(1, c->kb.NPI) * sizeof(cplx<T>)) != hipSuccess ||
        hipMalloc((void**)&y.kbv, (size_t)c->NKB * std::max(1, c->kb.NT) * sizeof(cplx<T>)) != hipSuccess ||
        hipMalloc((void**)&y.rows, (size_t)c->NKB * 8 * sizeof(double)) != hipSuccess)
      return bfail(b, SALMON_ERR_NOMEM, "batch buffers (system %d)", i);
    b->bufs.push_back(y.uv);
    b->bufs.push_back(y.ph);
    b->bufs.push_back(y.phn);
    b->bufs.push_back(y.kbv);
    b->bufs.push_back(y.rows);
    b->max_ph = std::max(b->max_ph, (long)c->NK * c->kb.NPI);
    y.pblk = (std::max(1, c->kb.Nlma) + 3) / 4;
    y.hblk = (c->g.NL / y.zb + 255) / 256;
    y.kblk = (c->kb.NT + 255) / 256;
    const long nb[kPhases] = {(long)c->NKB * y.pblk, 0, (long)((nv + 255) / 256), (long)c->NKB,
                              (long)c->NKB * y.kblk};
    for (int ph = 0; ph < kPhases; ++ph) {
      if (ph == 1) continue;
      y.first[ph] = acc[ph];
      acc[ph] += nb[ph];
    }
    y.first[kPhases] = 0;
  }
  // stencil blocks class by class, so that one launch per z blocking covers
  // every system of the class
  const int zbs[4] = {1, 2, 4, 8};
  for (int k = 0; k < 4 && !b->resident; ++k) {
    b->zcls[k][0] = acc[1];
    for (int i = 0; i < n; ++i) {
      if (S[i].zb != zbs[k]) continue;
      S[i].first[1] = acc[1];
      acc[1] += (long)S[i].NKB * S[i].hblk;
    }
    b->zcls[k][1] = acc[1] - b->zcls[k][0];
  }
  for (int ph = 0; ph < kPhases && !b->resident; ++ph) {
    b->first[ph].assign(1, acc[ph]);
    std::vector<unsigned short> own((size_t)acc[ph]);
    for (int i = 0; i < n; ++i) {
      const long cnt = ph == 0 ? (long)S[i].NKB * S[i].pblk
                     : ph == 1 ? (long)S[i].NKB * S[i].hblk
                     : ph == 2 ? (long)(((size_t)S[i].NKB * S[i].g.NL + 255) / 256)
                     : ph == 3 ? (long)S[i].NKB : (long)S[i].NKB * S[i].kblk;
      std::fill(own.begin() + S[i].first[ph], own.begin() + S[i].first[ph] + cnt, (unsigned short)i);
    }
    if (hipMalloc((void**)&b->d_owner[ph], sizeof(unsigned short) * std::max<size_t>(1, own.size())) != hipSuccess)
      return bfail(b, SALMON_ERR_NOMEM, "batch block tables");
    b->bufs.push_back(b->d_owner[ph]);
    BHIP(b, hipMemcpy(b->d_owner[ph], own.data(), sizeof(unsigned short) * own.size(), hipMemcpyHostToDevice));
  }
  if (!b->d_next) {
    BHIP(b, hipMalloc((void**)&b->d_next, 2 * sizeof(int)));
    BHIP(b, hipMemset(b->d_next, 0, 2 * sizeof(int)));
  }
  b->sweep = b->resident;
  if (!b->resident && (r = sweep_plan<T>(b, S))) return r;
  if (hipMalloc(&b->d_sys, sizeof(Sys<T>) * n) != hipSuccess) return bfail(b, SALMON_ERR_NOMEM, "batch descriptors");
  b->bufs.push_back(b->d_sys);
  BHIP(b, hipMemcpy(b->d_sys, S.data(), sizeof(Sys<T>) * n, hipMemcpyHostToDevice));
  b->ready = true;
  return SALMON_OK;
}

// One launch of the persistent sweep, its phases (`which`, see k_b_phase; layers = 2:
// also those of which = 2) and work queue before it.
template <typename T>
static void batch_sweep_launch(salmon_batch* b, const Sys<T>* S, const Step& st, int which, int layers) {
  hipLaunchKernelGGL(k_b_begin<T>, dim3((unsigned)std::max(1L, (b->max_ph + 255) / 256), (unsigned)b->ctx.size(), layers),
                     dim3(256), 0, b->stream, S, st, which, b->d_next);
  if constexpr (sizeof(T) == 4)
    hipLaunchKernelGGL((k_b_sweep<T, 4>), dim3(b->sweep_grid), dim3(sweep_waves<T>() * kWave), b->sweep_lds, b->stream,
                       S, st, (const int2*)b->d_items, b->nitems, b->d_next);
  else
    hipLaunchKernelGGL((k_b_sweep<T, 2>), dim3(b->sweep_grid), dim3(sweep_waves<T>() * kWave), b->sweep_lds, b->stream,
                       S, st, (const int2*)b->d_items, b->nitems, b->d_next);
}

// One step's launches (captured by batch_run).
template <typename T>
static int batch_enqueue_step(salmon_batch* b, double dt, long ac_stride) {
  const int n = (int)b->ctx.size();
  const Sys<T>* S = (const Sys<T>*)b->d_sys;
  const Step st{b->d_ac, b->d_step, dt, {b->d_owner[0], b->d_owner[1], b->d_owner[2], b->d_owner[3], b->d_owner[4]},
                ac_stride};
  if (b->sweep) {
    // the step's launch also forms the previous step's observables (at
    // A(t_n)), whose rows the sum then takes
    batch_sweep_launch<T>(b, S, st, 0, 2);
    hipLaunchKernelGGL(k_b_sum<T>, dim3(n), dim3(256), 0, b->stream, S, n, b->d_step, b->d_res, 1, 1,
                       (unsigned*)b->d_next + 1);
    BHIP(b, hipGetLastError());
    return SALMON_OK;
  }
  if (b->max_ph > 0)
    hipLaunchKernelGGL(k_b_phase<T>, dim3((unsigned)((b->max_ph + 255) / 256), n), dim3(256), 0, b->stream, S, st, 0);
  for (int t = 0; t < 4; ++t) {
    hipLaunchKernelGGL(k_b_project<T>, dim3((unsigned)b->first[0][0]), dim3(256), 0, b->stream, S, n, t, st);
    if (b->first[4][0] > 0)
      hipLaunchKernelGGL(k_b_kbapply<T>, dim3((unsigned)b->first[4][0]), dim3(256), 0, b->stream, S, st);
    if (b->zcls[0][1]) hipLaunchKernelGGL((k_b_hpsi<T, 1>), dim3((unsigned)b->zcls[0][1]), dim3(256), 0, b->stream, S, t, st, b->zcls[0][0]);
    if (b->zcls[1][1]) hipLaunchKernelGGL((k_b_hpsi<T, 2>), dim3((unsigned)b->zcls[1][1]), dim3(256), 0, b->stream, S, t, st, b->zcls[1][0]);
    if (b->zcls[2][1]) hipLaunchKernelGGL((k_b_hpsi<T, 4>), dim3((unsigned)b->zcls[2][1]), dim3(256), 0, b->stream, S, t, st, b->zcls[2][0]);
    if (b->zcls[3][1]) hipLaunchKernelGGL((k_b_hpsi<T, 8>), dim3((unsigned)b->zcls[3][1]), dim3(256), 0, b->stream, S, t, st, b->zcls[3][0]);
  }
  hipLaunchKernelGGL(k_b_fold<T>, dim3((unsigned)b->first[2][0]), dim3(256), 0, b->stream, S, n, st);
  // the observables' phases at k + A(t+dt) (the step's projections are done)
  if (b->max_ph > 0)
    hipLaunchKernelGGL(k_b_phase<T>, dim3((unsigned)((b->max_ph + 255) / 256), n), dim3(256), 0, b->stream, S, st, 1);
  hipLaunchKernelGGL(k_b_observe<T>, dim3((unsigned)b->first[3][0]), dim3(256), 0, b->stream, S, n, st);
  hipLaunchKernelGGL(k_b_sum<T>, dim3(n), dim3(256), 0, b->stream, S, n, b->d_step, b->d_res, 0, 1,
                     (unsigned*)b->d_next + 1);
  BHIP(b, hipGetLastError());
  return SALMON_OK;
}

// Descriptors of the batch whose k tables are kbase[i] (system i's device
// kAc(NK,3) table, in place of its kAc0 + A), a zero A(t) table and a zero
// step counter, built on the first call for a kbase array and kept with the
// work buffers.
template <typename T>
static int batch_k_descriptors(salmon_batch* b, const double* const* kbase) {
  const int n = (int)b->ctx.size();
  int r;
  if (!b->tuned && (r = batch_tune<T>(b))) return r;
  if (!b->sweep) return bfail(b, SALMON_ERR_UNSUPPORTED, "the persistent sweep is not set up");
  if (b->d_sys_k && b->sys_k_base == kbase) return SALMON_OK;
  if (!b->d_sys_k) {
    if (hipMalloc(&b->d_sys_k, sizeof(Sys<T>) * n) != hipSuccess ||
        hipMalloc((void**)&b->d_zero_ac, sizeof(double) * 6) != hipSuccess ||
        hipMalloc((void**)&b->d_zero_step, sizeof(int)) != hipSuccess)
      return bfail(b, SALMON_ERR_NOMEM, "batch k descriptors");
    b->bufs.push_back(b->d_sys_k);
    b->bufs.push_back(b->d_zero_ac);
    b->bufs.push_back(b->d_zero_step);
    BHIP(b, hipMemsetAsync(b->d_zero_ac, 0, sizeof(double) * 6, b->stream));
    BHIP(b, hipMemsetAsync(b->d_zero_step, 0, sizeof(int), b->stream));
  }
  std::vector<Sys<T>> S(n);
  BHIP(b, hipMemcpyAsync(S.data(), b->d_sys, sizeof(Sys<T>) * n, hipMemcpyDeviceToHost, b->stream));
  BHIP(b, hipStreamSynchronize(b->stream));
  for (int i = 0; i < n; ++i) S[i].kac0 = kbase[i];
  BHIP(b, hipMemcpyAsync(b->d_sys_k, S.data(), sizeof(Sys<T>) * n, hipMemcpyHostToDevice, b->stream));
  BHIP(b, hipStreamSynchronize(b->stream));
  b->sys_k_base = kbase;
  return SALMON_OK;
}

// One Taylor-4 step (hamiltonian.f90:27-123) of every orbital of the batch at
// the k points kbase[i] over dt, without observables: the persistent sweep
// with the step counter at 0 (so no observables are formed) and A = 0.
template <typename T>
static int batch_taylor(salmon_batch* b, const double* const* kbase, double dt) {
  const int n = (int)b->ctx.size();
  int r;
  if ((r = batch_k_descriptors<T>(b, kbase))) return r;
  const Sys<T>* S = (const Sys<T>*)b->d_sys_k;
  if (b->resident) return resident_launch<T>(b, S, ResArgs{nullptr, 0L, 0, 1, dt, 1, 0}, nullptr);
  const Step st{b->d_zero_ac, b->d_zero_step, dt,
                {b->d_owner[0], b->d_owner[1], b->d_owner[2], b->d_owner[3], b->d_owner[4]}, 0L};
  batch_sweep_launch<T>(b, S, st, 0, 1);
  BHIP(b, hipGetLastError());
  return SALMON_OK;
}

// The observables rows' sums of every system's orbitals at the k points
// kbase[i] (current.f90, total_energy.f90 terms and the norm, as k_b_sum lays
// them out) into out (nsys x 8): one observables-only sweep launch.
template <typename T>
static int batch_observe(salmon_batch* b, const double* const* kbase, double* out) {
  const int n = (int)b->ctx.size();
  int r;
  if ((r = batch_k_descriptors<T>(b, kbase))) return r;
  if (b->cap_steps < 1 || !b->d_res) {
    if (b->d_res) (void)hipFree(b->d_res);
    b->d_res = nullptr;
    BHIP(b, hipMalloc((void**)&b->d_res, sizeof(double) * 8 * (size_t)n));
    b->cap_steps = 1;
    if (b->exec) (void)hipGraphExecDestroy(b->exec);  // the step graph holds the old results pointer
    b->exec = nullptr;
  }
  const Sys<T>* S = (const Sys<T>*)b->d_sys_k;
  if (b->resident) {
    if ((r = resident_launch<T>(b, S, ResArgs{nullptr, 0L, 0, 1, 0.0, 0, 1}, b->d_res))) return r;
  } else {
    const Step st{b->d_zero_ac, b->d_zero_step, 0.0,
                  {b->d_owner[0], b->d_owner[1], b->d_owner[2], b->d_owner[3], b->d_owner[4]}, 0L, 1};
    batch_sweep_launch<T>(b, S, st, 2, 1);
    hipLaunchKernelGGL(k_b_sum<T>, dim3(n), dim3(256), 0, b->stream, S, n, b->d_zero_step, b->d_res, 0, 0,
                       (unsigned*)nullptr);
    BHIP(b, hipGetLastError());
  }
  BHIP(b, hipMemcpyAsync(out, b->d_res, sizeof(double) * 8 * (size_t)n, hipMemcpyDeviceToHost, b->stream));
  BHIP(b, hipStreamSynchronize(b->stream));
  return SALMON_OK;
}

// After the last step of a run on the persistent sweep: the observables of
// the final orbitals (at A(t_nsteps), the device counter then holding nsteps)
// into the run's last result row.
template <typename T>
static int batch_close_sweep(salmon_batch* b, double dt, long ac_stride) {
  const int n = (int)b->ctx.size();
  const Sys<T>* S = (const Sys<T>*)b->d_sys;
  const Step st{b->d_ac, b->d_step, dt, {b->d_owner[0], b->d_owner[1], b->d_owner[2], b->d_owner[3], b->d_owner[4]},
                ac_stride, 1};
  batch_sweep_launch<T>(b, S, st, 2, 1);
  hipLaunchKernelGGL(k_b_sum<T>, dim3(n), dim3(256), 0, b->stream, S, n, b->d_step, b->d_res, 1, 0, (unsigned*)nullptr);
  BHIP(b, hipGetLastError());
  return SALMON_OK;
}

// Times the stencil launch of system i alone for each z blocking that divides NLz.
template <typename T>
static int batch_tune_one(salmon_batch* b, int i, int* best) {
  salmon_ctx* c = b->ctx[i];
  std::vector<Sys<T>> one(1);
  BHIP(b, hipMemcpy(one.data(), (Sys<T>*)b->d_sys + i, sizeof(Sys<T>), hipMemcpyDeviceToHost));
  Sys<T>* d1 = nullptr;
  BHIP(b, hipMalloc((void**)&d1, sizeof(Sys<T>)));
  hipEvent_t e0, e1;
  BHIP(b, hipEventCreate(&e0));
  BHIP(b, hipEventCreate(&e1));
  float bestt = 1e30f;
  *best = 1;
  // the single-system launch below addresses blocks 0.. of a one-system table
  std::vector<unsigned short> zeros((size_t)one[0].NKB * ((c->g.NL + 255) / 256) + 1, 0);
  unsigned short* d_zero = nullptr;
  BHIP(b, hipMalloc((void**)&d_zero, sizeof(unsigned short) * zeros.size()));
  BHIP(b, hipMemcpy(d_zero, zeros.data(), sizeof(unsigned short) * zeros.size(), hipMemcpyHostToDevice));
  const Step st{b->d_ac, b->d_step, 0.0, {d_zero, d_zero, d_zero, d_zero, d_zero}, 0};
  for (int zb : {1, 2, 4, 8}) {
    if (c->g.NLz % zb) continue;
    Sys<T> y = one[0];
    y.zb = zb;
    y.hblk = (c->g.NL / zb + 255) / 256;
    y.first[1] = 0;
    BHIP(b, hipMemcpy(d1, &y, sizeof(Sys<T>), hipMemcpyHostToDevice));
    if ((long)y.NK * y.kb.NPI > 0)
      hipLaunchKernelGGL(k_b_phase<T>, dim3((unsigned)(((long)y.NK * y.kb.NPI + 255) / 256), 1), dim3(256), 0, b->stream,
                         (const Sys<T>*)d1, st, 0);
    const unsigned nblk = (unsigned)((long)y.NKB * y.hblk);
    float tmin = 1e30f;
    for (int rep = 0; rep < 4; ++rep) {
      BHIP(b, hipEventRecord(e0, b->stream));
      switch (zb) {
        case 1: hipLaunchKernelGGL((k_b_hpsi<T, 1>), dim3(nblk), dim3(256), 0, b->stream, (const Sys<T>*)d1, 0, st, 0L); break;
        case 2: hipLaunchKernelGGL((k_b_hpsi<T, 2>), dim3(nblk), dim3(256), 0, b->stream, (const Sys<T>*)d1, 0, st, 0L); break;
        case 4: hipLaunchKernelGGL((k_b_hpsi<T, 4>), dim3(nblk), dim3(256), 0, b->stream, (const Sys<T>*)d1, 0, st, 0L); break;
        default: hipLaunchKernelGGL((k_b_hpsi<T, 8>), dim3(nblk), dim3(256), 0, b->stream, (const Sys<T>*)d1, 0, st, 0L); break;
      }
      BHIP(b, hipEventRecord(e1, b->stream));
      BHIP(b, hipEventSynchronize(e1));
      float ms = 0;
      BHIP(b, hipEventElapsedTime(&ms, e0, e1));
      if (rep > 0) tmin = std::min(tmin, ms);
    }
    if (tmin < bestt) {
      bestt = tmin;
      *best = zb;
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  (void)hipFree(d1);
  (void)hipFree(d_zero);
  return SALMON_OK;
}

template <typename T>
static int batch_tune(salmon_batch* b) {
  // build with z blocking 1 first (work buffers and descriptors for timing)
  batch_release(b);
  b->zb.assign(b->ctx.size(), 1);
  int r = batch_build<T>(b);
  if (r) return r;
  if (!b->d_step) {
    BHIP(b, hipMalloc((void**)&b->d_step, sizeof(int)));
    BHIP(b, hipMemset(b->d_step, 0, sizeof(int)));
  }
  if (!b->d_ac) {
    BHIP(b, hipMalloc((void**)&b->d_ac, sizeof(double) * 6));
    BHIP(b, hipMemset(b->d_ac, 0, sizeof(double) * 6));
    b->cap_ac = 6;
  }
  BHIP(b, hipMemset(b->d_step, 0, sizeof(int)));
  if (b->sweep) {  // the persistent sweep chooses its column shapes without timing
    b->tuned = true;
    return SALMON_OK;
  }
  std::vector<std::array<int, 4>> shapes;  // (NLx, NLy, NLz, zb)
  std::vector<int> zb(b->ctx.size(), 1);
  for (size_t i = 0; i < b->ctx.size(); ++i) {
    const Grid& g = b->ctx[i]->g;
    int found = -1;
    for (size_t j = 0; j < shapes.size(); ++j)
      if (shapes[j][0] == g.NLx && shapes[j][1] == g.NLy && shapes[j][2] == g.NLz) found = (int)j;
    if (found < 0) {
      int best = 1;
      if ((r = batch_tune_one<T>(b, (int)i, &best))) return r;
      shapes.push_back({g.NLx, g.NLy, g.NLz, best});
      found = (int)shapes.size() - 1;
    }
    zb[i] = shapes[found][3];
  }
  batch_release(b);
  b->zb = zb;
  b->tuned = true;
  return batch_build<T>(b);
}

// nsteps steps; ac is one A(t) table (nsteps+1, 3) for every system, or
// (per_sys) one per system, (nsys, nsteps+1, 3)
template <typename T>
static int batch_run(salmon_batch* b, const double* ac, int nsteps, double dt, double* jt, double* et, double* norm,
                     bool per_sys) {
  const int n = (int)b->ctx.size();
  int r;
  if (!b->tuned && (r = batch_tune<T>(b))) return r;
  const size_t need_ac = (size_t)3 * (nsteps + 1) * (per_sys ? n : 1);
  const long stride = per_sys ? 3L * (nsteps + 1) : 0L;
  if (need_ac > b->cap_ac || !b->d_ac) {
    if (b->d_ac) (void)hipFree(b->d_ac);
    b->d_ac = nullptr;
    BHIP(b, hipMalloc((void**)&b->d_ac, sizeof(double) * need_ac));
    b->cap_ac = need_ac;
    if (b->exec) (void)hipGraphExecDestroy(b->exec);  // the graph holds the old table pointer
    b->exec = nullptr;
  }
  if ((size_t)nsteps > b->cap_steps || !b->d_res) {
    if (b->d_res) (void)hipFree(b->d_res);
    b->d_res = nullptr;
    BHIP(b, hipMalloc((void**)&b->d_res, sizeof(double) * 8 * (size_t)n * nsteps));
    b->cap_steps = nsteps;
    if (b->exec) (void)hipGraphExecDestroy(b->exec);
    b->exec = nullptr;
  }
  BHIP(b, hipMemcpyAsync(b->d_ac, ac, sizeof(double) * need_ac, hipMemcpyHostToDevice, b->stream));
  // a resident batch: kResSteps steps per launch, straight from the A(t) tables
  if (b->resident)
    for (int s = 0; s < nsteps; s += kResSteps) {
      const ResArgs a{b->d_ac, stride, s, std::min(kResSteps, nsteps - s), dt, 1, 1};
      if ((r = resident_launch<T>(b, (const Sys<T>*)b->d_sys, a, b->d_res))) return r;
    }
  const bool graph_steps = !b->resident;
  if (graph_steps) BHIP(b, hipMemsetAsync(b->d_step, 0, sizeof(int), b->stream));
  if (b->exec && (b->graph_dt != dt || b->graph_stride != stride)) {
    (void)hipGraphExecDestroy(b->exec);
    b->exec = nullptr;
  }
  if (graph_steps && !b->exec) {
    hipGraph_t graph = nullptr;
    BHIP(b, hipStreamBeginCapture(b->stream, hipStreamCaptureModeRelaxed));
    r = batch_enqueue_step<T>(b, dt, stride);
    const hipError_t e = hipStreamEndCapture(b->stream, &graph);
    if (r) {
      if (graph) (void)hipGraphDestroy(graph);
      return r;
    }
    if (e != hipSuccess) return bfail(b, SALMON_ERR_HIP, "step capture: %s", hipGetErrorString(e));
    const hipError_t ei = hipGraphInstantiate(&b->exec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    if (ei != hipSuccess) return bfail(b, SALMON_ERR_HIP, "step graph: %s", hipGetErrorString(ei));
    b->graph_dt = dt;
    b->graph_stride = stride;
  }
  if (graph_steps)
    for (int s = 0; s < nsteps; ++s) BHIP(b, hipGraphLaunch(b->exec, b->stream));
  if (graph_steps && b->sweep && (r = batch_close_sweep<T>(b, dt, stride))) return r;
  std::vector<double> res(8 * (size_t)n * nsteps);
  BHIP(b, hipMemcpyAsync(res.data(), b->d_res, sizeof(double) * res.size(), hipMemcpyDeviceToHost, b->stream));
  BHIP(b, hipStreamSynchronize(b->stream));
  for (int i = 0; i < n; ++i)
    for (int s = 0; s < nsteps; ++s) {
      const double* q = &res[((size_t)s * n + i) * 8];
      if (jt)
        for (int d = 0; d < 3; ++d) jt[((size_t)i * nsteps + s) * 3 + d] = q[d];
      if (et) et[(size_t)i * nsteps + s] = q[3] + q[4] + q[5];
      if (norm) norm[(size_t)i * nsteps + s] = q[6];
    }
  return SALMON_OK;
}
