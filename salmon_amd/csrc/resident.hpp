// LDS-resident orbitals: whole RT steps of one orbital per workgroup, for the
// systems of a batch (and single contexts off 16^3) whose orbital fits in LDS.
//
// The persistent sweep (batch_sweep.hpp) streams each orbital through global
// memory with one barrier per x plane; on small grids its planes hold less work
// than their latency (a 12^3 step of 12 orbitals took 100 us, 1.2 us per plane).
// Here a workgroup of up to 12 waves reads its orbital into LDS once, and every
// H application is two barriers: all threads take the 24 neighbours of their
// points from LDS into registers while the atoms' KB terms are formed (one wave
// per atom), then every point adds its KB term and becomes the next input in
// place.  Orbitals do not depend on each other while the potential is frozen, so
// one launch runs all the steps of a run, observables included, and its k
// points' phases are formed in the workgroup: no launch per step.
//
// Measured per step of a 10-step run (FP64 / complex64, us; the sweep before): 8^3
// x 4 orbitals 23 / 22 (76 / 67), 12^3 x 4 36 / 30 (151 / 161), 16^3 x 256
// 66 / 47 (278 / 334), 16^3 x 1024 225 / 158 (337 / 376).  What bounds it is the
// latency of the chain barrier - LDS reads - KB reduction - barrier; at 16^3 the
// 24 LDS reads per point (FP64: 768 cycles per 64 points at 128 bytes per cycle).
//
// Layout: a wave owns 64 columns of the (y,z) plane at PX consecutive x, so LDS
// accesses are to consecutive values and the x neighbours' planes are
// wave-uniform.  PX is the smallest that 12 waves cover the grid with (most
// threads per point, for latency).
#pragma once
#include "batch.hpp"

namespace salmon {
namespace batch {

constexpr int kResMaxWaves = 12;  // three per SIMD: 168 vector registers each
constexpr size_t kResMaxLds = 160 * 1024 - 256;
constexpr int kResLpa = 4;  // projectors per atom

// x points per thread for the grid: the smallest of the compiled ones whose waves
// fit a workgroup, or 0
inline int res_px(const Grid& g) {
  const int ncb = (g.NLy * g.NLz + kWave - 1) / kWave;
  for (int px : {1, 2, 3, 4, 6})
    if (ncb * ((g.NLx + px - 1) / px) <= kResMaxWaves) return px;
  return 0;
}
inline int res_waves(const Grid& g, int px) {
  return (g.NLy * g.NLz + kWave - 1) / kWave * ((g.NLx + px - 1) / px);
}
// LDS: the orbital; per sphere point the KB term (with a zero entry), the phases
// at the Taylor and the observables' k, the projector values and the grid index;
// per-axis phase tables, per-wave sums, per-atom tables
template <typename T>
inline size_t res_lds(const Grid& g, int NPI, int NI) {
  const size_t n1 = ((size_t)NPI + 4) / 4 * 4;
  return sizeof(cplx<double>) * 10 * (size_t)(g.NLx + g.NLy + g.NLz) + sizeof(cplx<T>) * ((size_t)g.NL + 3 * n1) +
         sizeof(double) * 10 * kResMaxWaves + sizeof(T) * kResLpa * (n1 + NI) + sizeof(int) * (n1 + NI + 1);
}

// Per-system tables of the resident kernel.
struct ResTab {
  gptr<const int> prim;      // (NL) first sphere point covering a grid point, or NPI
  gptr<const int> code;      // (NPI) px | py << 10 | pz << 20 into the per-axis phase tables
  gptr<const double> uvp;    // (NPI, kResLpa) uV(j, l) of the sphere point's atom, zero past its projectors
  gptr<const double> sgp;    // (NI, kResLpa) iuV
  gptr<const int> ov_start;  // (nov+1) grid points inside several spheres: entries
  gptr<const int> ov_jp;     // [ov_start[o]+1, ov_start[o+1]) of ov_jp add into ov_jp[ov_start[o]]
  int nov;
  double cc[3][4], dc[3][4];  // -lap(n)/2 and nab(n) per axis, n = 1..4
};

struct ResArgs {
  const double* ac;       // A(t) rows (system s at s * ac_stride), or null: A = 0
  long ac_stride;
  int n0, nsteps;         // steps n0 .. n0 + nsteps - 1
  double dt;
  int taylor, obs;        // what each step does: the Taylor step, the observables after it
};

// A complex64 coefficient in a vector register: an FP32 instruction with a
// scalar operand holds its SIMD for 4.2 cycles, one with vector operands for 2.4
// to 3 (measured on the MI355X, two or more waves per SIMD).
__device__ __forceinline__ float vector_reg(float v) {
  asm volatile("" : "+v"(v));
  return v;
}
__device__ __forceinline__ double vector_reg(double v) { return v; }

// The value is complete here: without it the optimiser sinks a result's
// arithmetic past the barrier to its use, and every neighbour value of every point
// stays in registers until then.
template <typename T>
__device__ __forceinline__ void pin(cplx<T>& v) {
  asm volatile("" : "+v"(v.re), "+v"(v.im));
}

template <typename T, int PX>
__global__ void __launch_bounds__(kResMaxWaves* kWave) k_b_resident(const Sys<T>* __restrict__ S,
                                                                    const ResTab* __restrict__ tabs,
                                                                    const int2* __restrict__ items, ResArgs a) {
  const int2 it = items[blockIdx.x];  // (system, orbital)
  const int s = __builtin_amdgcn_readfirstlane(it.x), o = __builtin_amdgcn_readfirstlane(it.y);
  const Sys<T>& y = S[s];
  const ResTab& rt = tabs[s];
  const Grid& g = y.g;
  const KBTables& kb = y.kb;
  const int NX = g.NLx, NY = g.NLy, NZ = g.NLz, NYZ = NY * NZ, NL = g.NL, NPI = kb.NPI, n1 = (NPI + 4) / 4 * 4;
  const int t = threadIdx.x, lane = t & (kWave - 1), NT = blockDim.x, NW = NT / kWave;
  const int wv = __builtin_amdgcn_readfirstlane(t / kWave);

  extern __shared__ __align__(16) unsigned char lds[];
  cplx<double>* ptab = (cplx<double>*)lds;
  cplx<T>* buf = (cplx<T>*)(ptab + 10 * (NX + NY + NZ));
  cplx<T>* dps = buf + NL;
  cplx<T>* em = dps + n1;
  cplx<T>* en = em + n1;
  double* red = (double*)(en + n1);
  T* ug = (T*)(red + 10 * kResMaxWaves);        // uV at [jp * kResLpa + l]
  T* fac = ug + kResLpa * n1;                   // Hxyz iuV per atom and projector
  int* gix = (int*)(fac + kResLpa * kb.NI);     // grid index of each sphere point
  int* ast = gix + n1;                          // first sphere point of each atom

  // the wave's columns and planes
  const int ncb = (NYZ + kWave - 1) / kWave;
  const int seg = __builtin_amdgcn_readfirstlane(wv / ncb), cb = wv - seg * ncb;
  const int x0 = seg * PX, cnt = min(PX, NX - x0);
  const bool act = cb * kWave + lane < NYZ;
  const int col = act ? cb * kWave + lane : 0;
  auto valid = [&](int i) { return act && i < cnt; };

  const int ik = o / y.NB;
  const double k0[3] = {y.kac0[ik], y.kac0[y.NK + ik], y.kac0[2 * y.NK + ik]};
  const double occ = y.occ[o];
  // LDS byte offsets, in plane x = 0, of the column and of its y and z neighbours (+1..+4, -1..-4)
  constexpr int kSz = sizeof(cplx<T>);
  const int base = 10 * (NX + NY + NZ) * (int)sizeof(cplx<double>);
  const int colb = base + col * kSz;
  int yo[8], zo[8];
  {
    const int iy = col / NZ, iz = col - iy * NZ;
#pragma unroll
    for (int n = 1; n <= 4; ++n) {
      yo[n - 1] = base + ((iy + n < NY ? iy + n : iy + n - NY) * NZ + iz) * kSz;
      yo[n + 3] = base + ((iy >= n ? iy - n : iy - n + NY) * NZ + iz) * kSz;
      zo[n - 1] = base + (iy * NZ + (iz + n < NZ ? iz + n : iz + n - NZ)) * kSz;
      zo[n + 3] = base + (iy * NZ + (iz >= n ? iz - n : iz - n + NZ)) * kSz;
    }
  }
  T cc[3][4], dc[3][4];
#pragma unroll
  for (int d = 0; d < 3; ++d)
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      cc[d][n] = vector_reg((T)rt.cc[d][n]);
      dc[d][n] = vector_reg((T)rt.dc[d][n]);
    }
  const double lap0 = g.lap[0][0] + g.lap[1][0] + g.lap[2][0];
  // per own point: the first sphere point covering it (16 bits each), the potential
  int prim[(PX + 1) / 2];
  T vf[PX];
  cplx<T> cur[PX], acc[PX];
  cplx<T>* zu = y.zu + (size_t)o * NL;
#pragma unroll
  for (int i = 0; i < PX; ++i) {
    const int p = (i < cnt ? x0 + i : x0) * NYZ + col;
    if (i % 2 == 0) prim[i / 2] = 0;
    prim[i / 2] |= (valid(i) ? rt.prim[p] : NPI) << (16 * (i & 1));
    vf[i] = y.vloc[p];
    cur[i] = zu[p];
  }
  if (t == 0) dps[NPI] = cplx<T>{0, 0};
  for (int q = t; q < NPI; q += NT) gix[q] = kb.pidx[q];
  for (int q = t; q < kResLpa * NPI; q += NT) ug[q] = (T)rt.uvp[q];
  for (int q = t; q < kResLpa * kb.NI; q += NT) fac[q] = (T)(g.Hxyz * rt.sgp[q]);
  for (int q = t; q <= kb.NI; q += NT) ast[q] = kb.atom_start[q];
  auto put = [&]() {
#pragma unroll
    for (int i = 0; i < PX; ++i)
      if (valid(i)) buf[(x0 + i) * NYZ + col] = cur[i];
  };
  // neighbour sums of own point i: L = sum_a sum_n (-lap_n/2)(psi+ + psi-),
  // G_a = sum_n nab_n (psi+ - psi-) (stencil/F90/hpsi.f90:190)
  auto sums = [&](int i, T& Lr, T& Li, T(&gr)[3], T(&gi)[3]) __attribute__((always_inline)) {
    int x = __builtin_amdgcn_readfirstlane(i < cnt ? x0 + i : x0);
    // opaque, so that the addresses are formed here and not kept in registers over all applications
    asm volatile("" : "+s"(x));
    auto at = [&](int plane, int off) { return *(const cplx<T>*)(lds + plane * (NYZ * kSz) + off); };
    Lr = Li = 0;
#pragma unroll
    for (int d = 0; d < 3; ++d) gr[d] = gi[d] = 0;
#pragma unroll
    for (int n = 1; n <= 4; ++n) {
      const int xp = x + n < NX ? x + n : x + n - NX, xm = x >= n ? x - n : x - n + NX;
      const cplx<T> q[6] = {at(x, zo[n - 1]), at(x, zo[n + 3]), at(x, yo[n - 1]), at(x, yo[n + 3]), at(xp, colb), at(xm, colb)};
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const cplx<T> p = q[4 - 2 * d], m = q[5 - 2 * d];
        Lr += cc[d][n - 1] * (p.re + m.re);
        Li += cc[d][n - 1] * (p.im + m.im);
        gr[d] += dc[d][n - 1] * (p.re - m.re);
        gi[d] += dc[d][n - 1] * (p.im - m.im);
      }
      if (n % 2 == 0) __builtin_amdgcn_sched_barrier(0);  // bounds the loads in flight by the register budget
    }
  };
  put();

  const T z1i = (T)(-a.dt), z2r = (T)(-a.dt * a.dt / 2.0), z3i = (T)(a.dt * a.dt * a.dt / 6.0),
          z4r = (T)(a.dt * a.dt * a.dt * a.dt / 24.0);
#pragma unroll 1
  for (int st = 0; st < a.nsteps; ++st) {
    double km[3], kn[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double* ac = a.ac ? a.ac + (size_t)s * a.ac_stride + 3 * (size_t)(a.n0 + st) : nullptr;
      km[d] = k0[d] + (ac ? 0.5 * (ac[d] + ac[3 + d]) : 0.0);
      kn[d] = k0[d] + (ac ? ac[3 + d] : 0.0);
    }
    // phases e^{ik.(r_j - T_j)} of the sphere points at both k, from per-axis
    // tables exp(i k_a (l H_a - j L_a)), l = 0..N_a-1, j = -2..2
    const int nph = 5 * (NX + NY + NZ);
    for (int q = t; q < 2 * nph; q += NT) {
      int r = q < nph ? q : q - nph, ax = 0, n = NX;
      if (r >= 5 * (NX + NY)) { ax = 2; n = NZ; r -= 5 * (NX + NY); }
      else if (r >= 5 * NX) { ax = 1; n = NY; r -= 5 * NX; }
      const int img = r / n, l = r - img * n;
      const double h = ax == 0 ? g.Hx : (ax == 1 ? g.Hy : g.Hz), L = ax == 0 ? g.aLx : (ax == 1 ? g.aLy : g.aLz);
      const double k = q < nph ? (ax == 0 ? km[0] : (ax == 1 ? km[1] : km[2]))
                               : (ax == 0 ? kn[0] : (ax == 1 ? kn[1] : kn[2]));
      double sn, cs;
      sincos(k * (l * h - (img - 2) * L), &sn, &cs);
      ptab[q] = cplx<double>{cs, sn};
    }
    __syncthreads();
    for (int q = t; q < 2 * NPI; q += NT) {
      const int jp = q < NPI ? q : q - NPI, c = rt.code[jp];
      const cplx<double>* tb = ptab + (q < NPI ? 0 : nph);
      const cplx<double> u = tb[c & 1023], v = tb[5 * NX + ((c >> 10) & 1023)], w = tb[5 * (NX + NY) + (c >> 20)];
      const cplx<double> uv{u.re * v.re - u.im * v.im, u.re * v.im + u.im * v.re};
      (q < NPI ? em : en)[jp] = cplx<T>{(T)(uv.re * w.re - uv.im * w.im), (T)(uv.re * w.im + uv.im * w.re)};
    }
    __syncthreads();
    if (a.taylor) {
      const T kx = (T)km[0], ky = (T)km[1], kz = (T)km[2];
      const T A = (T)((km[0] * km[0] + km[1] * km[1] + km[2] * km[2] - lap0) * 0.5);
#pragma unroll
      for (int i = 0; i < PX; ++i) acc[i] = cur[i];
#pragma unroll 1
      for (int n = 0; n < 4; ++n) {
        // KB term of pseudo_pt (hpsi.f90:176-206), a wave per atom:
        //   U(l) = Hxyz iuV(l) sum_j uV(j,l) e^{ik.r_j} psi(J_j),  dps(j) = e^{-ik.r_j} sum_l uV(j,l) U(l)
        for (int at = wv; at < kb.NI; at += NW) {
          const int j0 = ast[at], m = ast[at + 1] - j0;
          if (m == 0) continue;
          T q[2 * kResLpa];
#pragma unroll
          for (int l = 0; l < 2 * kResLpa; ++l) q[l] = 0;
          for (int jb = 0; jb < m; jb += 2 * kWave) {
            cplx<T> e[2], v[2];
            T u[2][kResLpa];
#pragma unroll
            for (int h = 0; h < 2; ++h) {  // two passes' loads in flight; past the sphere: its first point, weight zero
              const int j = jb + h * kWave + lane, jp = j0 + (j < m ? j : 0);
              e[h] = em[jp];
              v[h] = buf[gix[jp]];
#pragma unroll
              for (int l = 0; l < kResLpa; ++l) u[h][l] = j < m ? ug[jp * kResLpa + l] : (T)0;
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const T wr = e[h].re * v[h].re - e[h].im * v[h].im, wi = e[h].re * v[h].im + e[h].im * v[h].re;
#pragma unroll
              for (int l = 0; l < kResLpa; ++l) {
                q[2 * l] += u[h][l] * wr;
                q[2 * l + 1] += u[h][l] * wi;
              }
            }
          }
          wave_sums(q);
          T sr[kResLpa], si[kResLpa];
#pragma unroll
          for (int l = 0; l < kResLpa; ++l) {
            const T f = fac[at * kResLpa + l];
            sr[l] = lane_read(q[0], wave_sums_lane(2 * l)) * f;
            si[l] = lane_read(q[0], wave_sums_lane(2 * l + 1)) * f;
          }
          for (int j = lane; j < m; j += kWave) {
            T tr = 0, ti = 0;
#pragma unroll
            for (int l = 0; l < kResLpa; ++l) {
              const T u = ug[(j0 + j) * kResLpa + l];
              tr += u * sr[l];
              ti += u * si[l];
            }
            const cplx<T> e = em[j0 + j];
            dps[j0 + j] = cplx<T>{e.re * tr + e.im * ti, e.re * ti - e.im * tr};  // conj(e) * t
          }
        }
#pragma unroll
        for (int i = 0; i < PX; ++i) {
          T Lr, Li, gr[3], gi[3];
          sums(i, Lr, Li, gr, gi);
          const cplx<T> e = cur[i];
          const T vA = vf[i] + A;
          cur[i].re = vA * e.re + Lr + (kx * gi[0] + ky * gi[1] + kz * gi[2]);
          cur[i].im = vA * e.im + Li - (kx * gr[0] + ky * gr[1] + kz * gr[2]);
          pin(cur[i]);
        }
        lds_barrier();  // every wave has read its inputs, every KB term is in LDS
        if (rt.nov > 0) {
          for (int q = t; q < rt.nov; q += NT) {
            const int q0 = rt.ov_start[q], q1 = rt.ov_start[q + 1];
            cplx<T> s0 = dps[rt.ov_jp[q0]];
            for (int r = q0 + 1; r < q1; ++r) {
              const cplx<T> d = dps[rt.ov_jp[r]];
              s0.re += d.re;
              s0.im += d.im;
            }
            dps[rt.ov_jp[q0]] = s0;
          }
          lds_barrier();
        }
        const T zr = (n == 1) ? z2r : ((n == 3) ? z4r : (T)0);
        const T zi = (n == 0) ? z1i : ((n == 2) ? z3i : (T)0);
#pragma unroll
        for (int i = 0; i < PX; ++i) {
          const cplx<T> d = dps[(prim[i / 2] >> (16 * (i & 1))) & 0xffff];
          const cplx<T> e{cur[i].re + d.re, cur[i].im + d.im};
          // one of zr, zi is zero: the zero one adds an exact zero
          acc[i].re = fma(zr, e.re, fma(-zi, e.im, acc[i].re));
          acc[i].im = fma(zr, e.im, fma(zi, e.re, acc[i].im));
          cur[i] = n < 3 ? e : acc[i];  // the fourth result only enters the Taylor sum
        }
        put();
        lds_barrier();
      }
    }
    if (a.obs) {
      // observables at kn, products and sums in FP64 (as in col_sweep and kb_observe_atom)
      double v[8] = {0, 0, 0, 0, 0, 0, 0, 0};  // |psi|^2, V|psi|^2, kinetic, current x, y, z
#pragma unroll
      for (int i = 0; i < PX; ++i) {
        T Lr, Li, gr[3], gi[3];
        sums(i, Lr, Li, gr, gi);
        const double er = valid(i) ? (double)cur[i].re : 0.0, ei = valid(i) ? (double)cur[i].im : 0.0;
        const double a2 = er * er + ei * ei;
        v[0] += a2;
        v[1] += (double)vf[i] * a2;
        v[2] += er * (double)Lr + ei * (double)Li;
#pragma unroll
        for (int d = 0; d < 3; ++d) v[3 + d] += er * (double)gi[d] - ei * (double)gr[d];
      }
      wave_sums(v);
#pragma unroll
      for (int i = 0; i < 6; ++i) {
        const double r = lane_read(v[0], wave_sums_lane(i));
        if (lane == 0) red[wv * 10 + i] = r;
      }
      // nonlocal current and energy (current.f90:247-269, total_energy.f90:191-199):
      // the projections U first; the current is then linear in the point terms,
      // r_j (Re w_j sum_l sg_l Im U_l uV(j,l) - Im w_j sum_l sg_l Re U_l uV(j,l)), w_j = e_j psi_j
      double nlj[3] = {0, 0, 0}, nle = 0;
      auto uv64 = [&](int jp, int l) -> double {  // complex64: not the values rounded to single
        if constexpr (sizeof(T) == 8) return ug[jp * kResLpa + l];
        else return rt.uvp[(size_t)jp * kResLpa + l];
      };
      for (int at = wv; at < kb.NI; at += NW) {
        const int j0 = ast[at], m = ast[at + 1] - j0;
        double q[2 * kResLpa];
#pragma unroll
        for (int l = 0; l < 2 * kResLpa; ++l) q[l] = 0;
        for (int j = lane; j < m; j += kWave) {
          const cplx<T> e = en[j0 + j], b = buf[gix[j0 + j]];
          const double wr = (double)e.re * b.re - (double)e.im * b.im, wi = (double)e.re * b.im + (double)e.im * b.re;
#pragma unroll
          for (int l = 0; l < kResLpa; ++l) {
            const double u = uv64(j0 + j, l);
            q[2 * l] += u * wr;
            q[2 * l + 1] += u * wi;
          }
        }
        wave_sums(q);
        double P[kResLpa], Q[kResLpa], e9 = 0;
#pragma unroll
        for (int l = 0; l < kResLpa; ++l) {
          const double ur = lane_read(q[0], wave_sums_lane(2 * l)), ui = lane_read(q[0], wave_sums_lane(2 * l + 1));
          const double sg = rt.sgp[at * kResLpa + l];
          P[l] = sg * ui;
          Q[l] = sg * ur;
          e9 += sg * (ur * ur + ui * ui);
        }
        double jm[4] = {0, 0, 0, 0};
        for (int j = lane; j < m; j += kWave) {
          const cplx<T> e = en[j0 + j], b = buf[gix[j0 + j]];
          const double wr = (double)e.re * b.re - (double)e.im * b.im, wi = (double)e.re * b.im + (double)e.im * b.re;
          double sa = 0, sb = 0;
#pragma unroll
          for (int l = 0; l < kResLpa; ++l) {
            const double u = uv64(j0 + j, l);
            sa += P[l] * u;
            sb += Q[l] * u;
          }
          const double cj = wr * sa - wi * sb;
#pragma unroll
          for (int d = 0; d < 3; ++d) jm[d] += kb.pos[3 * (size_t)(j0 + j) + d] * cj;
        }
        wave_sums(jm);
#pragma unroll
        for (int d = 0; d < 3; ++d) nlj[d] += lane_read(jm[0], wave_sums_lane(d));
        nle += e9;
      }
      if (lane == 0) {
#pragma unroll
        for (int d = 0; d < 3; ++d) red[wv * 10 + 6 + d] = nlj[d];
        red[wv * 10 + 9] = nle;
      }
      __syncthreads();
      if (t == 0) {
        double r[10];
#pragma unroll
        for (int i = 0; i < 10; ++i) {
          r[i] = 0;
          for (int w = 0; w < NW; ++w) r[i] += red[w * 10 + i];
        }
        const double hx = g.Hxyz, sc = hx / g.aLxyz;
        double* row = y.rrows + ((size_t)st * y.NKB + o) * 8;
#pragma unroll
        for (int d = 0; d < 3; ++d)
          row[d] = occ * (kn[d] * r[0] + r[3 + d]) * sc + occ / g.aLxyz * 2.0 * hx * hx * r[6 + d];
        row[3] = occ * (-0.5 * lap0 * r[0] + r[2] + kn[0] * r[3] + kn[1] * r[4] + kn[2] * r[5]) * hx +
                 occ * (kn[0] * kn[0] + kn[1] * kn[1] + kn[2] * kn[2]) / 2.0;
        row[4] = occ * hx * hx * r[9];
        row[5] = occ * r[1] * hx;
        row[6] = occ * r[0] * hx;
        row[7] = 0.0;
      }
      __syncthreads();
    }
  }
  if (a.taylor) {
#pragma unroll
    for (int i = 0; i < PX; ++i)
      if (valid(i)) zu[(x0 + i) * NYZ + col] = cur[i];
  }
}

// Sums of the rows of step n0 + blockIdx.y of system blockIdx.x into res(step, system, 0..7).
template <typename T>
__global__ void __launch_bounds__(256) k_b_resident_sum(const Sys<T>* __restrict__ S, int n0, double* __restrict__ res) {
  __shared__ double smem[4 * 8];
  const Sys<T>& y = S[blockIdx.x];
  const double* rows = y.rrows + (size_t)blockIdx.y * y.NKB * 8;
  double v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int r = threadIdx.x; r < y.NKB; r += 256) {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] += rows[(size_t)r * 8 + i];
  }
  block_sum256<8>(v, smem);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int i = 0; i < 8; ++i) res[((size_t)(n0 + blockIdx.y) * gridDim.x + blockIdx.x) * 8 + i] = v[i];
  }
}

}  // namespace batch
}  // namespace salmon
