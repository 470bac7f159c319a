// Self-consistent local potential of the RT step (ARTED/RT/dt_evolve.f90:
// 185-207 with no_update_func = 'n'): from the density rho(t+dt), the Hartree
// potential (ARTED/common/Hartree.f90:20-128: rho(G), V_H(G) = 4 pi rho(G)/|G|^2
// without G = 0, and back, in the three launches of dft.hpp) and the
// PZ81 LDA exchange-correlation potential (src/xc/builtin_pz.f90:24-80 as
// called by src/xc/salmon_xc.f90:499-511), Vloc = V_H + Vpsl + V_xc.
// Orthorhombic cells.  FP64 throughout; the complex64 orbitals' potential copy
// is refreshed from the FP64 one.
#pragma once
#include "dft.hpp"

namespace salmon {
namespace scf {

constexpr int kMaxN = 256;  // points per axis of the DFT passes (twiddle table rows)

// rho(x; y, z) to its z and y transforms.  Grid (blocks of z lines, NLx).
__global__ void __launch_bounds__(256) k_rho_zy(const double* __restrict__ rho, cplx<double>* __restrict__ f, Grid g,
                                                int nl, const double* __restrict__ tw) {
  const size_t o = (size_t)blockIdx.y * g.NLy * g.NLz;
  dft::plane<true>(g.NLz, g.NLy, nl, tw + 4 * kMaxN, tw + 2 * kMaxN, -1.0,
                   [&](int z, int y) { return cplx<double>{rho[o + y * g.NLz + z], 0.0}; },
                   [&](int z, int y, cplx<double> v) { f[o + y * g.NLz + z] = v; });
}

// The x transform, 4 pi / |G|^2 / NL with G = 0 dropped, and back along x.
__global__ void __launch_bounds__(256) k_coulomb_x(cplx<double>* __restrict__ f, Grid g, const double* __restrict__ tw) {
  dft::lines_x(g, f, tw, [&](int ix, int iy, int iz) {
    const int nx = ix < g.NLx - g.NLx / 2 ? ix : ix - g.NLx;
    const int ny = iy < g.NLy - g.NLy / 2 ? iy : iy - g.NLy;
    const int nz = iz < g.NLz - g.NLz / 2 ? iz : iz - g.NLz;
    const double pi = 3.141592653589793;
    const double gx = 2.0 * pi * nx / g.aLx, gy = 2.0 * pi * ny / g.aLy, gz = 2.0 * pi * nz / g.aLz;
    const double G2 = gx * gx + gy * gy + gz * gz;
    return (nx == 0 && ny == 0 && nz == 0) ? 0.0 : 4.0 * pi / G2 / g.NL;
  });
}

// PZ81 e_xc and its density derivative at the total density t (with the
// reference's + 1e-10 and its branch at rs = 1); returns v_xc.
__device__ __forceinline__ double pz_vxc(double rho) {
  const double pi = 3.141592653589793;
  const double gU = -0.1423, b1U = 1.0529, b2U = 0.3334, AU = 0.0311, BU = -0.048, CU = 0.002, DU = -0.0116;
  const double cst = 0.75 * pow(3.0 / (2.0 * pi), 2.0 / 3.0);
  const double t = rho + 1e-10;
  const double rs = pow(3.0 / (4.0 * pi * t), 1.0 / 3.0);
  double e = -cst / rs, de = e / (3.0 * t);
  if (rs > 1.0) {
    const double q = sqrt(rs), den = 1.0 + b1U * q + b2U * rs;
    e += gU / den;
    de += gU * (0.5 * b1U * q + b2U * rs) / (3.0 * t) / (den * den);
  } else {
    const double ln = log(rs);
    e += AU * ln + BU + CU * rs * ln + DU * rs;
    de -= rs / (3.0 * t) * (AU / rs + CU * (ln + 1.0) + DU);
  }
  return e + rho * de;
}

// V_H from its x-back-transformed rows by the y and z transforms, and Vloc = V_H +
// Vpsl + V_xc into the FP64 potential and its FP32 copy; vh/vxc (nullable) get the
// parts.  Grid (blocks of y lines, NLx).
__global__ void __launch_bounds__(256) k_vloc_yz(const cplx<double>* __restrict__ f, Grid g, int nl, const double* __restrict__ tw,
                                                 const double* __restrict__ rho, const double* __restrict__ vpsl, int xc,
                                                 double* __restrict__ v64, float* __restrict__ v32,
                                                 double* __restrict__ vh, double* __restrict__ vxc) {
  const size_t o = (size_t)blockIdx.y * g.NLy * g.NLz;
  dft::plane<false>(g.NLy, g.NLz, nl, tw + 2 * kMaxN, tw + 4 * kMaxN, 1.0,
                    [&](int y, int z) { return f[o + y * g.NLz + z]; },
                    [&](int y, int z, cplx<double> r) {
                      const size_t p = o + y * g.NLz + z;
                      const double h = r.re, x = xc ? pz_vxc(rho[p]) : 0.0;
                      const double v = h + (vpsl ? vpsl[p] : 0.0) + x;
                      v64[p] = v;
                      if (v32) v32[p] = (float)v;
                      if (vh) vh[p] = h;
                      if (vxc) vxc[p] = x;
                    });
}

// ETRS potential extrapolation (dt_evolve.f90:247-251): Vnew = 3 V - 3 V_old1 +
// V_old2, the history shifts (old2 <- old1, old1 <- V) and V <- Vnew with its
// FP32 copy
__global__ void __launch_bounds__(256) k_vloc_extrapolate(double* __restrict__ v64, float* __restrict__ v32,
                                                          double* __restrict__ old1, double* __restrict__ old2,
                                                          int NL) {
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p >= NL) return;
  const double v = v64[p], o1 = old1[p];
  const double vn = 3.0 * v - 3.0 * o1 + old2[p];
  old2[p] = o1;
  old1[p] = v;
  v64[p] = vn;
  v32[p] = (float)vn;
}

}  // namespace scf
}  // namespace salmon
