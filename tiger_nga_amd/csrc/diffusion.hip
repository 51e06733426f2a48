// Molar-diffusion correction of finite-rate chemistry on the GPU (gfx950):
// the body of finitechem_diffusion (reference combustion/finitechem.f90:538-923)
// and the source update of finitechem_source_transport (492-528).
//
// Stencil work over the caller's Fortran-layout fields, one lane per cell
// (i fastest, so every field and operator access of a wave is coalesced):
//   diff_cell_kernel  every cell of the ghosted block: mixture molar mass
//                     W_gp (finitechem_W) and heat capacity cp_mix (cv when
//                     compressible / constant volume);
//   diff_face_kernel  every face cell of the stencil range: the correction
//                     velocities corr_vel_{x,y,z} = sum over species of the
//                     Fickian (and molar) face fluxes;
//   diff_main_kernel  every interior cell: per species the corrected flux at
//                     the faces the divergence needs (recomputed per cell
//                     instead of stored: HBM-bound work, the recomputation
//                     is cheap arithmetic on cached neighbours), the species
//                     term div F_k, the enthalpy flux cp_k(T) interp_m(F_k)
//                     grad_m(T), the H2O / CO / CO2 dump, gas radiation, the
//                     cp-gradient term, / cp, * dt, and the optional update of
//                     the transport source.
// Second order has a pair of its own (diff_face2_kernel, diff_main2_kernel), and
// fourth order stores the face fluxes (diff_vel_kernel and the two after it).
// Readings where the reference text does not conform (the CPU oracle's too):
// SC(i-st2:j+st1) at 652 read as i+st1; the z sections k-st2:k-st1 at
// 634-635 and 706 read as k-st2:k+st1 (identical at second order); Cp_sp(isc)
// at 720-730 read as the species' own cp.  The burner heat loss (796-802) and
// the external ignition source (842-859) belong to single cases' meshes and
// are left to the caller.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "chem_device.h"
#include "chem_kernels.h"

namespace tgr {

namespace {

__device__ __forceinline__ int64_t c3(const DiffGeom& g, int i, int j, int k) {
  return (int64_t)(i - g.imino_) + (int64_t)g.nxo * ((int64_t)(j - g.jmino_) + (int64_t)g.nyo * (k - g.kmino_));
}

__device__ __forceinline__ bool wall(const DiffGeom& g, const int* mask, int i, int j) {
  return mask && mask[(i - g.imino) + (int64_t)g.mx * (j - g.jmino)] == 1;
}

// operator coefficient (i, j, st), first index from i0 (ni entries), second
// from j0 (nj), stencil from s0
__device__ __forceinline__ double op(const double* a, int i, int i0, int ni, int j, int j0, int nj, int st, int s0) {
  return a[(int64_t)(i - i0) + (int64_t)ni * ((int64_t)(j - j0) + (int64_t)nj * (st - s0))];
}

// thermo row (range, coefficient) of species k from the mechanism table block
__device__ __forceinline__ void cp_species(const char* tab, const TabLayout& L, double tmid, double T, int k,
                                           double& cp) {
  const double* c = (const double*)(tab + L.th + (T > tmid ? 0 : 13 * kRow)) + k;
  const int r = kRow / 8;
  const double ac = c[7 * r], d1 = c[8 * r], d2 = c[9 * r], d3 = c[10 * r], d4 = c[11 * r], d5 = c[12 * r];
  cp = ac * (d1 + T * (d2 + T * (d3 + T * (d4 + T * d5))));
}

}  // namespace

// Order of the workgroups: each takes consecutive cells of the range in storage
// order, whatever its extents, so that a block one cell wide fills its waves like
// a cube (GRI-3.0, second order, 1 x 1 x 4096 cells: 565 us with every plane
// rounded up to whole workgroups, 55 this way; 35 x 35 x 200: 224 and 154).  The
// workgroups of a plane, `row`, are taken kStrip at a time through all planes, then the next
// kStrip; the hardware deals workgroups to the 8 XCDs in turn, so XCD e (blockIdx
// % 8) takes the e-th eighth of that order: its resident workgroups cover a brick
// of kStrip workgroups by some 16 planes, whose halo is a third of its volume
// (GRI-3.0 128^3: 1610 us in plain order, 1504 in this one).
constexpr int kXcd = 8, kStrip = 4;
struct Cells {
  int ni, nj;         // extents of the range
  unsigned n, wg;     // its cells and workgroups
  unsigned row;       // workgroups of a plane (rounded: the bricks lean a little)
  unsigned threads;   // of a workgroup
  int k0;             // first plane of the range
  int64_t base;       // cells of the block before the ones that 32-bit offsets reach
};

__device__ __forceinline__ bool range_cell(const Cells& c, int& i, int& j, int& k) {
  const unsigned e = blockIdx.x % kXcd, first = (unsigned)((uint64_t)e * c.wg / kXcd),
                 last = (unsigned)((uint64_t)(e + 1) * c.wg / kXcd), seq = first + blockIdx.x / kXcd;
  unsigned w = seq;
  const unsigned rows = c.row ? c.wg / c.row : 0;  // whole rows; the cells past them follow in plain order
  if (seq < rows * c.row) {
    const unsigned whole = c.row / kStrip * kStrip, strip = seq / (rows * kStrip) * kStrip;
    const unsigned s0 = strip < whole ? strip : whole, width = strip < whole ? kStrip : c.row - whole;
    const unsigned r = seq - s0 * rows;
    w = r / width * c.row + s0 + r % width;
  }
  const unsigned q = w * blockDim.x + threadIdx.x, r = q / (unsigned)c.ni;
  i = (int)(q - r * (unsigned)c.ni);
  j = (int)(r % (unsigned)c.nj);
  k = c.k0 + (int)(r / (unsigned)c.nj);
  return seq < last && q < c.n;
}

// the cell of the face range / of the interior that this thread has
template <int ST1, int ST2>
__device__ __forceinline__ bool face_cell(const DiffParams& p, const Cells& cl, int& i, int& j, int& k) {
  const bool in = range_cell(cl, i, j, k);
  i += p.gm.imin_ - ST1;
  j += p.gm.jmin_ - ST1;
  k += p.gm.kmin_ - ST1;
  return in;
}

__device__ __forceinline__ bool interior_cell(const DiffParams& p, const Cells& cl, int& i, int& j, int& k) {
  const bool in = range_cell(cl, i, j, k);
  i += p.gm.imin_;
  j += p.gm.jmin_;
  k += p.gm.kmin_;
  return in;
}

// a[byte offset]: a wave-uniform base and a 32-bit lane offset (the launcher
// keeps the cells that a launch reaches below 2^32 bytes)
__device__ __forceinline__ double ldo(const double* a, unsigned off) {
  return *(const double*)((const char*)a + off);
}

// cp rows of the species in LDS, [species][T > tmid][6]
template <int NEQ>
__device__ __forceinline__ void stage_cp(double* cps, const char* tab) {
  constexpr TabLayout L = tab_layout<NEQ>();
  for (int t = threadIdx.x; t < (NEQ - 1) * 12; t += blockDim.x) {
    const int k = t / 12, hi = (t / 6) % 2, c = t % 6;
    cps[t] = *(const double*)(tab + L.th + (hi ? 0 : 13 * kRow) + (7 + c) * kRow + k * 8);
  }
  __syncthreads();
}

__device__ __forceinline__ double cp_lds(const double* c, double T) {
  return c[0] * (c[1] + T * (c[2] + T * (c[3] + T * (c[4] + T * c[5]))));
}

template <int NEQ>
__global__ __launch_bounds__(256) void diff_cell_kernel(DiffParams p) {
  constexpr TabLayout L = tab_layout<NEQ>();
  constexpr int N = NEQ - 1;
  __shared__ __attribute__((aligned(16))) double cps[N * 12];
  stage_cp<NEQ>(cps, p.mech.tab);
  const DiffGeom& g = p.gm;
  const int64_t n = (int64_t)g.nxo * g.nyo * g.nzo;
  const TGR_CONST double* W = (const TGR_CONST double*)(p.mech.tab + L.w);
  for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < n; c += (int64_t)gridDim.x * blockDim.x) {
    const int i = g.imino_ + (int)(c % g.nxo), j = g.jmino_ + (int)((c / g.nxo) % g.nyo);
    double w = 1.0, cp = 0.0;
    if (!wall(g, p.mask, i, j)) {
      const double T = p.sc[(int64_t)g.isc_T0 * g.plane + c];
      const double* Y = p.sc + (int64_t)g.isc_sc0 * g.plane + c;
      const double* cr = cps + (T > p.mech.tmid ? 6 : 0);
      double s1 = 0.0, s2 = 0.0;
#pragma unroll 4
      for (int k = 0; k < N; ++k) {
        const double yk = Y[k * g.plane];
        const double y = fmin(fmax(yk, 0.0), 1.0);
        s1 += y;
        s2 += y / W[k];
        cp += yk * cp_lds(cr + k * 12, T);
      }
      w = s1 / s2;
      if (p.cv) cp = cp - 8314.34 / w;
    }
    p.wg[c] = w;
    p.cpm[c] = cp;
  }
}

template <int NEQ>
__global__ __launch_bounds__(256) void diff_face_kernel(DiffParams p) {
  constexpr int N = NEQ - 1;
  const DiffGeom& g = p.gm;
  const tgr_metric_dev& m = p.m;
  const int st1 = m.st1, st2 = m.st2;
  const int fi0 = g.imin_ - st1, fni = g.imax_ + st2 - fi0 + 1;
  const int fj0 = g.jmin_ - st1, fnj = g.jmax_ + st2 - fj0 + 1;
  const int fk0 = g.kmin_ - st1, fnk = g.kmax_ + st2 - fk0 + 1;
  const int64_t n = (int64_t)fni * fnj * fnk;
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (int64_t)gridDim.x * blockDim.x) {
    const int i = fi0 + (int)(q % fni), j = fj0 + (int)((q / fni) % fnj), k = fk0 + (int)(q / ((int64_t)fni * fnj));
    const int64_t o = c3(g, i, j, k);
    double vx = 0.0, vy = 0.0, vz = 0.0;
    if (!wall(g, p.mask, i, j)) {
      for (int sp = 0; sp < N; ++sp) {
        const double* Y = p.sc + (int64_t)(g.isc_sc0 + sp) * g.plane;
        const double* D = p.diff + (int64_t)(g.isc_sc0 + sp) * g.plane;
        double a = 0, b = 0, a2 = 0, b2 = 0, a3 = 0, b3 = 0;
        double ix = 0, gx = 0, iy = 0, gy = 0, iz = 0, gz = 0;
        for (int s = -st2; s <= st1; ++s) {
          const int64_t ox = c3(g, i + s, j, k), oy = c3(g, i, j + s, k), oz = c3(g, i, j, k + s);
          const double wx = op(m.interp_sc_x, i, fi0, fni, j, g.jmino_, g.nyo, s, -st2);
          const double wy = op(m.interp_sc_y, i, g.imino_, g.nxo, j, fj0, fnj, s, -st2);
          const double wz = op(m.interp_sc_z, i, g.imino_, g.nxo, j, fj0, fnj, s, -st2);
          const double ggx = op(m.grad_x, i, fi0, fni, j, fj0, fnj, s, -st2);
          const double ggy = op(m.grad_y, i, fi0, fni, j, fj0, fnj, s, -st2);
          const double ggz = op(m.grad_z, i, fi0, fni, j, fj0, fnj, s, -st2);
          a += wx * D[ox];
          b += ggx * Y[ox];
          a2 += wy * D[oy];
          b2 += ggy * Y[oy];
          a3 += wz * D[oz];
          b3 += ggz * Y[oz];
          if (p.molar) {
            ix += wx * (Y[ox] / p.wg[ox]);
            gx += ggx * p.wg[ox];
            iy += wy * (Y[oy] / p.wg[oy]);
            gy += ggy * p.wg[oy];
            iz += wz * (Y[oz] / p.wg[oz]);
            gz += ggz * p.wg[oz];
          }
        }
        vx += a * b;
        vy += a2 * b2;
        vz += a3 * b3;
        if (p.molar) {
          vx += a * ix * gx;
          vy += a2 * iy * gy;
          vz += a3 * iz * gz;
        }
      }
    }
    p.cvel[o] = vx;
    p.cvel[g.plane + o] = vy;
    p.cvel[2 * g.plane + o] = vz;
  }
}

namespace {

// Corrected (and molar) flux and Fickian flux of species sp at the face
// cell (i, j, k) in direction d (0 x, 1 y, 2 z); 0 at a wall face.
struct Flux {
  double corr, fick;
};

__device__ __forceinline__ Flux face_flux(const DiffParams& p, int d, int i, int j, int k, const double* Y,
                                          const double* D) {
  const DiffGeom& g = p.gm;
  const tgr_metric_dev& m = p.m;
  if (wall(g, p.mask, i, j)) return {0.0, 0.0};
  const int st1 = m.st1, st2 = m.st2;
  const int fi0 = g.imin_ - st1, fni = g.imax_ + st2 - fi0 + 1;
  const int fj0 = g.jmin_ - st1, fnj = g.jmax_ + st2 - fj0 + 1;
  double sy = 0, a = 0, b = 0, iyw = 0, gw = 0;
  for (int s = -st2; s <= st1; ++s) {
    const int64_t o = d == 0 ? c3(g, i + s, j, k) : (d == 1 ? c3(g, i, j + s, k) : c3(g, i, j, k + s));
    const double w = d == 0 ? op(m.interp_sc_x, i, fi0, fni, j, g.jmino_, g.nyo, s, -st2)
                            : op(d == 1 ? m.interp_sc_y : m.interp_sc_z, i, g.imino_, g.nxo, j, fj0, fnj, s, -st2);
    const double gg = op(d == 0 ? m.grad_x : (d == 1 ? m.grad_y : m.grad_z), i, fi0, fni, j, fj0, fnj, s, -st2);
    sy += w * Y[o];
    a += w * D[o];
    b += gg * Y[o];
    if (p.molar) {
      iyw += w * (Y[o] / p.wg[o]);
      gw += gg * p.wg[o];
    }
  }
  Flux f;
  f.corr = -p.cvel[(int64_t)d * g.plane + c3(g, i, j, k)] * sy;
  if (p.molar) f.corr += a * iyw * gw;
  f.fick = a * b;
  return f;
}

// Gas radiation of the temperature equation (finitechem.f90:738-792):
// optically thin loss of H2O, CO2, CH4 and CO with the reference's Planck-mean
// absorption fits, Tb = 298 K; a species the mechanism lacks contributes 0.
__device__ __forceinline__ double gas_radiation(const DiffParams& p, double T, int64_t o) {
  const DiffGeom& g = p.gm;
  const double tm1 = 1000.0 / T;
  const double T2 = T * T;
  const double aH2O =
      -0.23093 + tm1 * (-1.12390 + tm1 * (9.41530 + tm1 * (-2.99880 + tm1 * (0.51382 + tm1 * -1.86840E-05))));
  const double aCO2 = 18.741 + tm1 * (-121.310 + tm1 * (273.500 + tm1 * (-194.050 + tm1 * (56.310 + tm1 * -5.8169))));
  const double aCH4 = 6.6334 - 0.0035686 * T + 1.6682e-08 * T2 + 2.5611e-10 * T2 * T - 2.6558e-14 * T2 * T2;
  const bool lo = T <= 750.0;
  const double aCO = lo ? 4.7869 + T * (-0.06953 + T * (2.95775e-4 + T * (-4.25732e-7 + T * 2.02894e-10)))
                        : 10.09 + T * (-0.01183 + T * (4.7753e-6 + T * (-5.87209e-10 + T * -2.5334e-14)));
  const double* S = p.sc;
  double sum = 0.0;
  if (p.i_co2 >= 0) sum += aCO2 * S[(int64_t)(g.isc_sc0 + p.i_co2) * g.plane + o] / p.w_co2;
  if (p.i_h2o >= 0) sum += aH2O * S[(int64_t)(g.isc_sc0 + p.i_h2o) * g.plane + o] / p.w_h2o;
  if (p.i_ch4 >= 0) sum += aCH4 * S[(int64_t)(g.isc_sc0 + p.i_ch4) * g.plane + o] / p.w_ch4;
  if (p.i_co >= 0) sum += aCO * S[(int64_t)(g.isc_sc0 + p.i_co) * g.plane + o] / p.w_co;
  const double radconst = 4.0 * 5.67051e-8 * 8314.34 / 101320.0;
  const double T4 = T2 * T2, Tb = 298.0;
  return -radconst * p.rho[o] * T * (T4 - Tb * Tb * Tb * Tb) * sum;
}

}  // namespace

template <int NEQ>
__global__ __launch_bounds__(256) void diff_main_kernel(DiffParams p) {
  constexpr TabLayout L = tab_layout<NEQ>();
  constexpr int N = NEQ - 1;
  const DiffGeom& g = p.gm;
  const tgr_metric_dev& m = p.m;
  const int st1 = m.st1, st2 = m.st2, stp = st1 + st2;
  const int nx = g.imax_ - g.imin_ + 1, ny = g.jmax_ - g.jmin_ + 1, nz = g.kmax_ - g.kmin_ + 1;
  const int64_t n = (int64_t)nx * ny * nz;
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (int64_t)gridDim.x * blockDim.x) {
    const int i = g.imin_ + (int)(q % nx), j = g.jmin_ + (int)((q / nx) % ny), k = g.kmin_ + (int)(q / ((int64_t)nx * ny));
    const int64_t o = c3(g, i, j, k);
    if (wall(g, p.mask, i, j)) continue;
    const int a0 = i - g.imin_, b0 = j - g.jmin_;
    const double* Tf = p.sc + (int64_t)g.isc_T0 * g.plane;
    const double T = Tf[o];
    // cell gradients of T and cp_mix
    double tx = 0, ty = 0, tz = 0, cx = 0, cy = 0, cz = 0;
    for (int s = -stp; s <= stp; ++s) {
      const double gxm = op(m.grad_xm, i, g.imin_, nx, j, g.jmin_, ny, s, -stp);
      const double gym = op(m.grad_ym, i, g.imin_, nx, j, g.jmin_, ny, s, -stp);
      const double gzm = op(m.grad_zm, i, g.imin_, nx, j, g.jmin_, ny, s, -stp);
      tx += gxm * Tf[c3(g, i + s, j, k)];
      ty += gym * Tf[c3(g, i, j + s, k)];
      tz += gzm * Tf[c3(g, i, j, k + s)];
      cx += gxm * p.cpm[c3(g, i + s, j, k)];
      cy += gym * p.cpm[c3(g, i, j + s, k)];
      cz += gzm * p.cpm[c3(g, i, j, k + s)];
    }
    double eT = 0.0;  // temperature term before the cp-gradient part and / cp
    for (int sp = 0; sp < N; ++sp) {
      const double* Y = p.sc + (int64_t)(g.isc_sc0 + sp) * g.plane;
      const double* D = p.diff + (int64_t)(g.isc_sc0 + sp) * g.plane;
      double dcor = 0.0, dfick = 0.0, fxm = 0.0, fym = 0.0, fzm = 0.0;
      for (int s = -st1; s <= st2; ++s) {
        const Flux fx = face_flux(p, 0, i + s, j, k, Y, D);
        const Flux fy = face_flux(p, 1, i, j + s, k, Y, D);
        const Flux fz = face_flux(p, 2, i, j, k + s, Y, D);
        const double du = op(m.div_u, i, g.imin_, nx, j, g.jmin_, ny, s, -st1);
        const double dv = op(m.div_v, i, g.imin_, nx, j, g.jmin_, ny, s, -st1);
        const double dw = op(m.div_w, i, g.imin_, nx, j, g.jmin_, ny, s, -st1);
        dcor += du * fx.corr + dv * fy.corr + dw * fz.corr;
        dfick += du * fx.fick + dv * fy.fick + dw * fz.fick;
        fxm += op(m.interp_u_xm, i, g.imin_, nx, j, g.jmin_, ny, s, -st1) * (fx.corr + fx.fick);
        fym += op(m.interp_v_ym, i, g.imin_, nx, j, g.jmin_, ny, s, -st1) * (fy.corr + fy.fick);
        fzm += op(m.interp_w_zm, i, g.imin_, nx, j, g.jmin_, ny, s, -st1) * (fz.corr + fz.fick);
      }
      double cpk;
      cp_species(p.mech.tab, L, p.mech.tmid, T, sp, cpk);
      eT = eT + cpk * fxm * tx;
      eT = eT + cpk * fym * ty;
      eT = eT + cpk * fzm * tz;
      if (p.corr) p.corr[(int64_t)sp * g.plane + o] = dcor * p.dt;
      if (p.src) p.src[(int64_t)(g.isc_sc0 + sp) * g.plane + o] += dcor * p.dt;
      if (p.dgp) {
        const int slot = sp == p.i_h2o ? 0 : (sp == p.i_co ? 1 : (sp == p.i_co2 ? 2 : -1));
        if (slot >= 0) p.dgp[(int64_t)slot * g.plane + o] = dfick + dcor;
      }
    }
    if (p.gasrad) eT += gas_radiation(p, T, o);
    const double dT = p.diff[(int64_t)g.isc_T0 * g.plane + o];
    eT = eT + dT * cx * tx;
    eT = eT + dT * cy * ty;
    eT = eT + dT * cz * tz;
    eT = eT / p.cpm[o] * p.dt;
    if (p.corr) p.corr[(int64_t)N * g.plane + o] = eT;
    if (p.src) p.src[(int64_t)g.isc_T0 * g.plane + o] += eT;
  }
}

// ---- second order (st1 = 0, st2 = 1) ----------------------------------------
// After diff_cell_kernel: diff_face2_kernel (the correction velocities, whose
// species sums the next pass needs complete) and diff_main2_kernel (the
// per-cell terms).  Both are bound by the rate at which the L1 serves the loads
// of Y and D (0.7 accesses per clock and CU, VALU busy 23 and 39 %): each species
// costs a cell 8 (14) of them and 50 (155) VALU instructions, so
//   * everything that does not depend on the species is formed before the
//     species loop (operator coefficients, w / W_gp, sum grad * W_gp, the
//     correction velocity), and the loop loads the next species while it
//     computes one;
//   * the cp coefficients are read from LDS, where the lanes of a wave differ
//     only in the temperature range;
//   * workgroups that share stencil planes run on the same XCD at the same
//     time (Cells above), so that the y and z neighbours are L2 hits.
// Every product and sum is rounded as the reference's text orders them (the
// molar factor apart: w (Y / W_gp) is (w / W_gp) Y).  Beside a wall, where W_gp
// jumps to 1, the molar fluxes of the species nearly cancel in the temperature
// term, and another order of the sums (the velocities' molar part summed apart,
// the divergence and enthalpy weights folded into the fluxes') moves single
// cells by up to 2.3e-12 of the field (2,000 random blocks).  GRI-3.0 128^3,
// molar term on: 2.37 -> 1.50 ms a call; in that other order 1.36.

// correction velocities at the face cells (diff_face_kernel; a face
// interpolates its cell and the one before it in each direction)
template <int NEQ, bool MOLAR>
__global__ __launch_bounds__(256) void diff_face2_kernel(DiffParams p, Cells cl) {
  constexpr int N = NEQ - 1;
  const DiffGeom& g = p.gm;
  const tgr_metric_dev& m = p.m;
  int i, j, k;
  if (!face_cell<0, 1>(p, cl, i, j, k)) return;
  const int fni = g.imax_ + 1 - g.imin_ + 1, fnj = g.jmax_ + 1 - g.jmin_ + 1;  // face range
  const int64_t o = c3(g, i, j, k);
  if (wall(g, p.mask, i, j)) {
    p.cvel[o] = p.cvel[g.plane + o] = p.cvel[2 * g.plane + o] = 0.0;
    return;
  }
  // coefficients of the two stencil points (s = -1, 0) per direction
  const int64_t step[3] = {1, g.nxo, (int64_t)g.nxo * g.nyo};
  double w[3][2], gg[3][2], wi[3][2], gw[3];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    w[0][t] = op(m.interp_sc_x, i, g.imin_, fni, j, g.jmino_, g.nyo, t - 1, -1);
    w[1][t] = op(m.interp_sc_y, i, g.imino_, g.nxo, j, g.jmin_, fnj, t - 1, -1);
    w[2][t] = op(m.interp_sc_z, i, g.imino_, g.nxo, j, g.jmin_, fnj, t - 1, -1);
    gg[0][t] = op(m.grad_x, i, g.imin_, fni, j, g.jmin_, fnj, t - 1, -1);
    gg[1][t] = op(m.grad_y, i, g.imin_, fni, j, g.jmin_, fnj, t - 1, -1);
    gg[2][t] = op(m.grad_z, i, g.imin_, fni, j, g.jmin_, fnj, t - 1, -1);
  }
  if constexpr (MOLAR) {
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double w0 = p.wg[o - step[d]], w1 = p.wg[o];
      gw[d] = 0.0;
      gw[d] += gg[d][0] * w0;
      gw[d] += gg[d][1] * w1;
      wi[d][0] = 1.0 / w0;
      wi[d][1] = 1.0 / w1;
    }
  }
  const unsigned oc = (unsigned)(o - cl.base) * 8u;
  const unsigned on[3] = {oc - 8u, oc - (unsigned)g.nxo * 8u, oc - (unsigned)g.nxo * (unsigned)g.nyo * 8u};
  const double* __restrict__ Y = p.sc + (int64_t)g.isc_sc0 * g.plane + cl.base;
  const double* __restrict__ D = p.diff + (int64_t)g.isc_sc0 * g.plane + cl.base;
  double yc = ldo(Y, oc), dc = ldo(D, oc), yn[3], dn[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) yn[d] = ldo(Y, on[d]), dn[d] = ldo(D, on[d]);
  double acc[3] = {0.0, 0.0, 0.0};
#pragma unroll 1
  for (int sp = 0; sp < N; ++sp) {
    const int64_t next = sp + 1 < N ? g.plane : 0;
    Y += next;
    D += next;
    const double yc2 = ldo(Y, oc), dc2 = ldo(D, oc);
    double yn2[3], dn2[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) yn2[d] = ldo(Y, on[d]), dn2[d] = ldo(D, on[d]);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      double a = 0, b = 0;
      a += w[d][0] * dn[d];
      b += gg[d][0] * yn[d];
      a += w[d][1] * dc;
      b += gg[d][1] * yc;
      acc[d] += a * b;
      if constexpr (MOLAR) {
        double ii = 0;
        ii += w[d][0] * (yn[d] * wi[d][0]);
        ii += w[d][1] * (yc * wi[d][1]);
        acc[d] += a * ii * gw[d];
      }
    }
    yc = yc2;
    dc = dc2;
#pragma unroll
    for (int d = 0; d < 3; ++d) yn[d] = yn2[d], dn[d] = dn2[d];
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) p.cvel[d * g.plane + o] = acc[d];
}

// What a face of a cell (diff_main_kernel: at the cell and the next one in each
// direction, each interpolating two cells) has that does not depend on the
// species: interpolation and gradient weights, -correction velocity, the molar
// term's w / W_gp and sum grad * W_gp.
struct FaceW {
  double w0, w1, g0, g1, v, u0, u1, gw;
};

// Y and D at a cell and its neighbours: the cell, then -, + in x, y, z
struct Stencil {
  double y[7], d[7];
};

__device__ __forceinline__ void load_stencil(Stencil& s, const double* Y, const double* D, unsigned oc, int64_t sy,
                                             int64_t sz) {
  s.y[0] = ldo(Y, oc), s.d[0] = ldo(D, oc);
  s.y[1] = ldo(Y - 1, oc), s.d[1] = ldo(D - 1, oc);
  s.y[2] = ldo(Y + 1, oc), s.d[2] = ldo(D + 1, oc);
  s.y[3] = ldo(Y - sy, oc), s.d[3] = ldo(D - sy, oc);
  s.y[4] = ldo(Y + sy, oc), s.d[4] = ldo(D + sy, oc);
  s.y[5] = ldo(Y - sz, oc), s.d[5] = ldo(D - sz, oc);
  s.y[6] = ldo(Y + sz, oc), s.d[6] = ldo(D + sz, oc);
}

template <int NEQ, bool MOLAR>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void diff_main2_kernel(DiffParams p, Cells cl) {
  constexpr int N = NEQ - 1;
  __shared__ __attribute__((aligned(16))) double cps[N * 12];
  stage_cp<NEQ>(cps, p.mech.tab);
  const DiffGeom& g = p.gm;
  int i, j, k;
  if (!interior_cell(p, cl, i, j, k)) return;
  const int nx = g.imax_ - g.imin_ + 1, ny = g.jmax_ - g.jmin_ + 1;
  const int fni = nx + 1, fnj = ny + 1;
  if (wall(g, p.mask, i, j)) return;
  const int64_t o = c3(g, i, j, k);
  const int64_t sy = g.nxo, sz = (int64_t)g.nxo * g.nyo;
  const int64_t step[3] = {1, sy, sz};
  const double* Tf = p.sc + (int64_t)g.isc_T0 * g.plane;
  const double T = Tf[o];
  // cell gradients of T and cp_mix (stp = 1)
  double tg[3] = {}, cg[3] = {};
#pragma unroll
  for (int s = -1; s <= 1; ++s)
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double* gm = d == 0 ? p.m.grad_xm : (d == 1 ? p.m.grad_ym : p.m.grad_zm);
      const double c = op(gm, i, g.imin_, nx, j, g.jmin_, ny, s, -1);
      tg[d] += c * Tf[o + s * step[d]];
      cg[d] += c * p.cpm[o + s * step[d]];
    }
  // wall faces carry no flux (the z faces of a non-wall cell are never walls)
  const bool live[3][2] = {{true, !wall(g, p.mask, i + 1, j)}, {true, !wall(g, p.mask, i, j + 1)}, {true, true}};
  FaceW fw[3][2];
  double dv[3][2], im[3][2];
#pragma unroll
  for (int d = 0; d < 3; ++d)
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      // the face cell is (i, j, k) + f along d; its two points are (-1, 0) for f = 0 and (0, +1) for f = 1
      FaceW& F = fw[d][f];
      const int fi = d == 0 ? i + f : i, fj = d == 1 ? j + f : j;
      const int64_t fo = o + f * step[d];
      if (d == 0) {
        F.w0 = op(p.m.interp_sc_x, fi, g.imin_, fni, fj, g.jmino_, g.nyo, -1, -1);
        F.w1 = op(p.m.interp_sc_x, fi, g.imin_, fni, fj, g.jmino_, g.nyo, 0, -1);
      } else {
        const double* ws = d == 1 ? p.m.interp_sc_y : p.m.interp_sc_z;
        F.w0 = op(ws, fi, g.imino_, g.nxo, fj, g.jmin_, fnj, -1, -1);
        F.w1 = op(ws, fi, g.imino_, g.nxo, fj, g.jmin_, fnj, 0, -1);
      }
      const double* gs = d == 0 ? p.m.grad_x : (d == 1 ? p.m.grad_y : p.m.grad_z);
      F.g0 = op(gs, fi, g.imin_, fni, fj, g.jmin_, fnj, -1, -1);
      F.g1 = op(gs, fi, g.imin_, fni, fj, g.jmin_, fnj, 0, -1);
      F.v = -p.cvel[d * g.plane + fo];
      if constexpr (MOLAR) {
        const double wa = p.wg[fo - step[d]], wb = p.wg[fo];
        F.u0 = F.w0 / wa;
        F.u1 = F.w1 / wb;
        F.gw = F.g0 * wa + F.g1 * wb;
      }
      const double* du = d == 0 ? p.m.div_u : (d == 1 ? p.m.div_v : p.m.div_w);
      const double* iu = d == 0 ? p.m.interp_u_xm : (d == 1 ? p.m.interp_v_ym : p.m.interp_w_zm);
      dv[d][f] = op(du, i, g.imin_, nx, j, g.jmin_, ny, f, 0);
      im[d][f] = op(iu, i, g.imin_, nx, j, g.jmin_, ny, f, 0);
    }
  const unsigned oc = (unsigned)(o - cl.base) * 8u;
  const double* __restrict__ Y = p.sc + (int64_t)g.isc_sc0 * g.plane + cl.base;
  const double* __restrict__ D = p.diff + (int64_t)g.isc_sc0 * g.plane + cl.base;
  const double* cr = cps + (T > p.mech.tmid ? 6 : 0);
  double* __restrict__ corr = p.corr;
  double* __restrict__ src = p.src;
  double* __restrict__ dgp = p.dgp;
  double eT = 0.0;  // temperature term before the cp-gradient part and / cp
  Stencil s;
  load_stencil(s, Y, D, oc, sy, sz);
#pragma unroll 1
  for (int sp = 0; sp < N; ++sp) {
    const int64_t next = sp + 1 < N ? g.plane : 0;
    Y += next;
    D += next;
    Stencil s2;
    load_stencil(s2, Y, D, oc, sy, sz);
    double dcor = 0.0, dfick = 0.0, fm[3] = {0.0, 0.0, 0.0};
    double fc[3][2], ff[3][2];
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        const FaceW& F = fw[d][f];
        const double y0 = f ? s.y[0] : s.y[2 * d + 1], y1 = f ? s.y[2 * d + 2] : s.y[0];
        const double d0 = f ? s.d[0] : s.d[2 * d + 1], d1 = f ? s.d[2 * d + 2] : s.d[0];
        double syf = 0, a = 0, b = 0;
        syf += F.w0 * y0;
        a += F.w0 * d0;
        b += F.g0 * y0;
        syf += F.w1 * y1;
        a += F.w1 * d1;
        b += F.g1 * y1;
        double c = F.v * syf;
        if constexpr (MOLAR) c += a * (F.u0 * y0 + F.u1 * y1) * F.gw;
        fc[d][f] = live[d][f] ? c : 0.0;
        ff[d][f] = live[d][f] ? a * b : 0.0;
      }
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      dcor += dv[0][f] * fc[0][f] + dv[1][f] * fc[1][f] + dv[2][f] * fc[2][f];
      dfick += dv[0][f] * ff[0][f] + dv[1][f] * ff[1][f] + dv[2][f] * ff[2][f];
#pragma unroll
      for (int d = 0; d < 3; ++d) fm[d] += im[d][f] * (fc[d][f] + ff[d][f]);
    }
    const double cpk = cp_lds(cr + sp * 12, T);
#pragma unroll
    for (int d = 0; d < 3; ++d) eT = eT + cpk * fm[d] * tg[d];
    if (corr) corr[(int64_t)sp * g.plane + o] = dcor * p.dt;
    if (src) src[(int64_t)(g.isc_sc0 + sp) * g.plane + o] += dcor * p.dt;
    if (dgp) {
      const int slot = sp == p.i_h2o ? 0 : (sp == p.i_co ? 1 : (sp == p.i_co2 ? 2 : -1));
      if (slot >= 0) dgp[(int64_t)slot * g.plane + o] = dfick + dcor;
    }
    s = s2;
  }
  if (p.gasrad) eT += gas_radiation(p, T, o);
  const double dT = p.diff[(int64_t)g.isc_T0 * g.plane + o];
#pragma unroll
  for (int d = 0; d < 3; ++d) eT = eT + dT * cg[d] * tg[d];
  eT = eT / p.cpm[o] * p.dt;
  if (corr) corr[(int64_t)N * g.plane + o] = eT;
  if (src) src[(int64_t)g.isc_T0 * g.plane + o] += eT;
}

// ---- wider stencils with widths known at compile time (fourth order) ----------
// After diff_cell_kernel: the correction velocities (diff_vel_kernel), every
// face's fluxes once per species into a workspace (diff_flux_kernel) and the
// cells' sums of them (diff_div_kernel), where diff_main_kernel has every cell
// recompute the fluxes of its 12 faces from 4 points each.  Every product and
// sum has the rounding that it has in the general kernels, so the outputs are
// theirs to the last bit (the molar quotients are divided, and the sums over the
// species run in their order: beside walls another order moves single cells by
// up to 2e-12 of the field).  A thread has a face of one direction (blockIdx.y):
// a species costs it eight loads and two stores, and a cell 24 loads, all along
// x; weights that do not depend on the species stay in registers.  The fluxes
// have no sum over the species, so those of a pass are split over blockIdx.z
// until there are six workgroups per CU.  The workspace holds nchunk species, one
// pass of them at a time.  The velocities are bound by FP64 (divisions; VALU 54 %
// busy) and L1 accesses (0.85 a clock and CU), the fluxes and their sums by the
// fluxes' way through memory (128 bytes per cell and species).
// DME39, 61 x 47 x 35 cells: 1144 (the general kernels) -> 309 us a call; GRI-3.0,
// 126 x 124 x 120: 18.4 -> 5.31 ms; DME39, 16 x 17 x 18: 830 -> 80 us (294 us, 4.30
// ms and 64 us with products for the quotients and the species' sums split over
// workgroups).

// Weights of the P = ST1 + ST2 + 1 stencil points of the faces in direction d.
template <int P>
struct Weights {
  double w[P], g[P], wg[P], gw;  // interpolation, gradient, W_gp, sum grad * W_gp
};

template <int ST1, int ST2, bool MOLAR>
__device__ __forceinline__ void face_weights(const DiffParams& p, int d, int i, int j, int64_t o, int64_t step,
                                             Weights<ST1 + ST2 + 1>& F) {
  const DiffGeom& g = p.gm;
  const tgr_metric_dev& m = p.m;
  const int fi0 = g.imin_ - ST1, fni = g.imax_ + ST2 - fi0 + 1, fj0 = g.jmin_ - ST1, fnj = g.jmax_ + ST2 - fj0 + 1;
  F.gw = 0.0;
#pragma unroll
  for (int t = 0; t < ST1 + ST2 + 1; ++t) {
    const int s = t - ST2;
    F.w[t] = d == 0 ? op(m.interp_sc_x, i, fi0, fni, j, g.jmino_, g.nyo, s, -ST2)
                    : op(d == 1 ? m.interp_sc_y : m.interp_sc_z, i, g.imino_, g.nxo, j, fj0, fnj, s, -ST2);
    F.g[t] = op(d == 0 ? m.grad_x : (d == 1 ? m.grad_y : m.grad_z), i, fi0, fni, j, fj0, fnj, s, -ST2);
    if constexpr (MOLAR) {
      F.wg[t] = p.wg[o + s * step];
      F.gw += F.g[t] * F.wg[t];
    }
  }
}

// Y and D of one species at the stencil points of a face
template <int ST1, int ST2>
struct FacePoints {
  double y[ST1 + ST2 + 1], d[ST1 + ST2 + 1];
  __device__ __forceinline__ void load(const double* Y, const double* D, unsigned oc, int64_t step) {
#pragma unroll
    for (int t = 0; t < ST1 + ST2 + 1; ++t) {
      y[t] = ldo(Y + (t - ST2) * step, oc);
      d[t] = ldo(D + (t - ST2) * step, oc);
    }
  }
};

template <int STP>
__device__ __forceinline__ void cell_gradient(const DiffParams& p, const double* f, int i, int j, int64_t o,
                                              double (&out)[3]) {
  const DiffGeom& g = p.gm;
  const int nx = g.imax_ - g.imin_ + 1, ny = g.jmax_ - g.jmin_ + 1;
  const int64_t step[3] = {1, g.nxo, (int64_t)g.nxo * g.nyo};
#pragma unroll
  for (int d = 0; d < 3; ++d) out[d] = 0.0;
#pragma unroll
  for (int s = -STP; s <= STP; ++s)
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double* gm = d == 0 ? p.m.grad_xm : (d == 1 ? p.m.grad_ym : p.m.grad_zm);
      out[d] += op(gm, i, g.imin_, nx, j, g.jmin_, ny, s, -STP) * f[o + s * step[d]];
    }
}

template <int NEQ, bool MOLAR, int ST1, int ST2>
__global__ __launch_bounds__(256) void diff_vel_kernel(DiffParams p, Cells cl) {
  constexpr int N = NEQ - 1, P = ST1 + ST2 + 1;
  const DiffGeom& g = p.gm;
  int i, j, k;
  if (!face_cell<ST1, ST2>(p, cl, i, j, k)) return;
  const int d = blockIdx.y;
  const int64_t o = c3(g, i, j, k), step = d == 0 ? 1 : (d == 1 ? g.nxo : (int64_t)g.nxo * g.nyo);
  double v = 0.0;
  if (!wall(g, p.mask, i, j)) {
    Weights<P> F;
    face_weights<ST1, ST2, MOLAR>(p, d, i, j, o, step, F);
    const unsigned oc = (unsigned)o * 8u;
    const double* __restrict__ Y = p.sc + (int64_t)g.isc_sc0 * g.plane;
    const double* __restrict__ D = p.diff + (int64_t)g.isc_sc0 * g.plane;
    FacePoints<ST1, ST2> s;
    s.load(Y, D, oc, step);
#pragma unroll 1
    for (int sp = 0; sp < N; ++sp) {
      const int64_t next = sp + 1 < N ? g.plane : 0;
      Y += next;
      D += next;
      FacePoints<ST1, ST2> s2;
      s2.load(Y, D, oc, step);
      double a = 0, b = 0, ii = 0;
#pragma unroll
      for (int t = 0; t < P; ++t) {
        a += F.w[t] * s.d[t];
        b += F.g[t] * s.y[t];
        if constexpr (MOLAR) ii += F.w[t] * (s.y[t] / F.wg[t]);
      }
      v += a * b;
      if constexpr (MOLAR) v += a * ii * F.gw;
      s = s2;
    }
  }
  p.cvel[d * g.plane + o] = v;
}

template <int NEQ, bool MOLAR, int ST1, int ST2>
__global__ __launch_bounds__(256) void diff_flux_kernel(DiffParams p, Cells cl, int sp0, int nsp) {
  constexpr int P = ST1 + ST2 + 1;
  const DiffGeom& g = p.gm;
  int i, j, k;
  if (!face_cell<ST1, ST2>(p, cl, i, j, k)) return;
  const int d = blockIdx.y;
  const int64_t o = c3(g, i, j, k), step = d == 0 ? 1 : (d == 1 ? g.nxo : (int64_t)g.nxo * g.nyo);
  // this workgroup's part of the species
  const int s0 = nsp * (int)blockIdx.z / (int)gridDim.z, s1 = nsp * ((int)blockIdx.z + 1) / (int)gridDim.z;
  if (s0 == s1) return;
  double* __restrict__ to = p.flux + (6 * s0 + 2 * d) * g.plane + o;
  if (wall(g, p.mask, i, j)) {  // no flux through a wall face
    for (int sp = s0; sp < s1; ++sp, to += 6 * g.plane) to[0] = to[g.plane] = 0.0;
    return;
  }
  Weights<P> F;
  face_weights<ST1, ST2, MOLAR>(p, d, i, j, o, step, F);
  const double v = -p.cvel[d * g.plane + o];
  const unsigned oc = (unsigned)o * 8u;
  const double* __restrict__ Y = p.sc + (int64_t)(g.isc_sc0 + sp0 + s0) * g.plane;
  const double* __restrict__ D = p.diff + (int64_t)(g.isc_sc0 + sp0 + s0) * g.plane;
  FacePoints<ST1, ST2> s;
  s.load(Y, D, oc, step);
#pragma unroll 1
  for (int sp = s0; sp < s1; ++sp, to += 6 * g.plane) {
    const int64_t next = sp + 1 < s1 ? g.plane : 0;
    Y += next;
    D += next;
    FacePoints<ST1, ST2> s2;
    s2.load(Y, D, oc, step);
    double yi = 0, a = 0, b = 0, ii = 0;
#pragma unroll
    for (int t = 0; t < P; ++t) {
      yi += F.w[t] * s.y[t];
      a += F.w[t] * s.d[t];
      b += F.g[t] * s.y[t];
      if constexpr (MOLAR) ii += F.w[t] * (s.y[t] / F.wg[t]);
    }
    double c = v * yi;
    if constexpr (MOLAR) c += a * ii * F.gw;
    to[0] = c;
    to[g.plane] = a * b;
    s = s2;
  }
}

template <int NEQ, int ST1, int ST2>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void diff_div_kernel(DiffParams p, Cells cl,
                                                                                               int sp0, int nsp) {
  constexpr int N = NEQ - 1, P = ST1 + ST2 + 1;
  __shared__ __attribute__((aligned(16))) double cps[N * 12];
  stage_cp<NEQ>(cps, p.mech.tab);
  const DiffGeom& g = p.gm;
  int i, j, k;
  if (!interior_cell(p, cl, i, j, k)) return;
  const int nx = g.imax_ - g.imin_ + 1, ny = g.jmax_ - g.jmin_ + 1;
  if (wall(g, p.mask, i, j)) return;
  const int64_t o = c3(g, i, j, k), step[3] = {1, g.nxo, (int64_t)g.nxo * g.nyo};
  const double* Tf = p.sc + (int64_t)g.isc_T0 * g.plane;
  const double T = Tf[o];
  double tg[3];
  cell_gradient<ST1 + ST2>(p, Tf, i, j, o, tg);
  double dv[3][P], im[3][P];
#pragma unroll
  for (int t = 0; t < P; ++t)
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double* a = d == 0 ? p.m.div_u : (d == 1 ? p.m.div_v : p.m.div_w);
      const double* b = d == 0 ? p.m.interp_u_xm : (d == 1 ? p.m.interp_v_ym : p.m.interp_w_zm);
      dv[d][t] = op(a, i, g.imin_, nx, j, g.jmin_, ny, t - ST1, -ST1);
      im[d][t] = op(b, i, g.imin_, nx, j, g.jmin_, ny, t - ST1, -ST1);
    }
  const double* cr = cps + (T > p.mech.tmid ? 6 : 0);
  const unsigned oc = (unsigned)o * 8u;
  const double* __restrict__ fl = p.flux;
  double eT = sp0 ? p.eT[o] : 0.0;  // temperature term of the species so far
#pragma unroll 1
  for (int sp = sp0; sp < sp0 + nsp; ++sp, fl += 6 * g.plane) {
    double fc[3][P], ff[3][P];
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
      for (int t = 0; t < P; ++t) {
        fc[d][t] = ldo(fl + 2 * d * g.plane + (t - ST1) * step[d], oc);
        ff[d][t] = ldo(fl + (2 * d + 1) * g.plane + (t - ST1) * step[d], oc);
      }
    double dcor = 0.0, dfick = 0.0, fm[3] = {};
#pragma unroll
    for (int t = 0; t < P; ++t) {
      dcor += dv[0][t] * fc[0][t] + dv[1][t] * fc[1][t] + dv[2][t] * fc[2][t];
      dfick += dv[0][t] * ff[0][t] + dv[1][t] * ff[1][t] + dv[2][t] * ff[2][t];
#pragma unroll
      for (int d = 0; d < 3; ++d) fm[d] += im[d][t] * (fc[d][t] + ff[d][t]);
    }
    const double cpk = cp_lds(cr + sp * 12, T);
#pragma unroll
    for (int d = 0; d < 3; ++d) eT = eT + cpk * fm[d] * tg[d];
    if (p.corr) p.corr[(int64_t)sp * g.plane + o] = dcor * p.dt;
    if (p.src) p.src[(int64_t)(g.isc_sc0 + sp) * g.plane + o] += dcor * p.dt;
    if (p.dgp) {
      const int slot = sp == p.i_h2o ? 0 : (sp == p.i_co ? 1 : (sp == p.i_co2 ? 2 : -1));
      if (slot >= 0) p.dgp[(int64_t)slot * g.plane + o] = dfick + dcor;
    }
  }
  if (sp0 + nsp < N) {
    p.eT[o] = eT;
    return;
  }
  double cg[3];
  cell_gradient<ST1 + ST2>(p, p.cpm, i, j, o, cg);
  if (p.gasrad) eT += gas_radiation(p, T, o);
  const double dT = p.diff[(int64_t)g.isc_T0 * g.plane + o];
#pragma unroll
  for (int d = 0; d < 3; ++d) eT = eT + dT * cg[d] * tg[d];
  eT = eT / p.cpm[o] * p.dt;
  if (p.corr) p.corr[(int64_t)N * g.plane + o] = eT;
  if (p.src) p.src[(int64_t)g.isc_T0 * g.plane + o] += eT;
}

// workgroups to launch: the same number for every XCD
unsigned launch_groups(const Cells& c) { return (c.wg + kXcd - 1) / kXcd * kXcd; }

template <int NEQ, bool MOLAR, int ST1, int ST2>
void launch_wide(const DiffParams& p, const Cells& cf, const Cells& cm, hipStream_t s) {
  const unsigned nf = launch_groups(cf);
  const dim3 gv(nf, 3), gf(nf, 3, p.nslice), gc(launch_groups(cm)), b(cf.threads), bc(cm.threads);
  hipLaunchKernelGGL((diff_vel_kernel<NEQ, MOLAR, ST1, ST2>), gv, b, 0, s, p, cf);
  for (int sp0 = 0; sp0 < NEQ - 1; sp0 += p.nchunk) {
    const int nsp = NEQ - 1 - sp0 < p.nchunk ? NEQ - 1 - sp0 : p.nchunk;
    hipLaunchKernelGGL((diff_flux_kernel<NEQ, MOLAR, ST1, ST2>), gf, b, 0, s, p, cf, sp0, nsp);
    hipLaunchKernelGGL((diff_div_kernel<NEQ, ST1, ST2>), gc, bc, 0, s, p, cm, sp0, nsp);
  }
}

}  // namespace tgr

using namespace tgr;

extern "C" int tgr_launch_diffusion(const DiffParams* p, int neq, hipStream_t s) {
  const DiffGeom& g = p->gm;
  const int64_t ncell = (int64_t)g.nxo * g.nyo * g.nzo;
  const int st1 = p->m.st1, st2 = p->m.st2;
  const int64_t nface = (int64_t)(g.imax_ - g.imin_ + 1 + st1 + st2) * (g.jmax_ - g.jmin_ + 1 + st1 + st2) *
                        (g.kmax_ - g.kmin_ + 1 + st1 + st2);
  const int64_t nint = (int64_t)(g.imax_ - g.imin_ + 1) * (g.jmax_ - g.jmin_ + 1) * (g.kmax_ - g.kmin_ + 1);
  auto blocks = [](int64_t n) { return (unsigned)std::min<int64_t>((n + 255) / 256, 65535); };
  // second order (the reference's default stencil) and fourth order have their
  // own kernels, which reach 2^29 cells by 32-bit byte offsets: second order
  // takes larger blocks by as many planes at a time (with the ones beside them)
  // as that allows; fourth order of larger blocks, and other widths, take the
  // general kernels
  const int64_t sz = (int64_t)g.nxo * g.nyo;
  const int slab = diff_small_plane(g.plane) ? g.nzo : (int)(((int64_t)1 << 29) / sz) - 2;
  const bool o2 = slab > 0 && st1 == 0 && st2 == 1, o4 = p->nchunk > 0;
  // planes [k0, k0 + slab) of the range that reaches `halo` cells past the interior
  auto range = [&](int halo, int k0, int slab) {
    const int ni = g.imax_ - g.imin_ + 1 + halo, nj = g.jmax_ - g.jmin_ + 1 + halo;
    const int nk = std::min(g.kmax_ - g.kmin_ + 1 + halo - k0, slab);
    const int64_t n = (int64_t)ni * nj * nk;
    // a wave per workgroup until every CU has four workgroups of four
    const int64_t t = n < (int64_t)4 * 256 * p->n_cu ? 64 : 256, row = ((int64_t)ni * nj + t / 2) / t;
    return Cells{ni, nj, (unsigned)n, (unsigned)((n + t - 1) / t), (unsigned)(row > kStrip ? row : 0), (unsigned)t,
                 k0, diff_small_plane(g.plane) ? 0 : (g.kmin_ + k0 - 1 - g.kmino_) * sz};
  };
  const int nz = g.kmax_ - g.kmin_ + 1;
  const Cells cm = range(0, 0, nz), cf = range(st1 + st2, 0, nz + st1 + st2);
#define TGR_DIFF_LAUNCH2(NEQ_, MOLAR_)                                                                              \
  hipLaunchKernelGGL(diff_cell_kernel<NEQ_>, dim3(blocks(ncell)), dim3(256), 0, s, *p);                           \
  for (int k0 = 0; k0 <= nz; k0 += slab) {                                                                          \
    const Cells c = range(1, k0, slab);                                                                             \
    hipLaunchKernelGGL((diff_face2_kernel<NEQ_, MOLAR_>), dim3(launch_groups(c)), dim3(c.threads), 0, s, *p, c);    \
  }                                                                                                                 \
  for (int k0 = 0; k0 < nz; k0 += slab) {                                                                           \
    const Cells c = range(0, k0, slab);                                                                             \
    hipLaunchKernelGGL((diff_main2_kernel<NEQ_, MOLAR_>), dim3(launch_groups(c)), dim3(c.threads), 0, s, *p, c);    \
  }
#define TGR_DIFF_LAUNCH(NEQ_)                                                                  \
  if (o2 && p->molar) {                                                                         \
    TGR_DIFF_LAUNCH2(NEQ_, true)                                                                \
  } else if (o2) {                                                                              \
    TGR_DIFF_LAUNCH2(NEQ_, false)                                                               \
  } else if (o4) {                                                                              \
    hipLaunchKernelGGL(diff_cell_kernel<NEQ_>, dim3(blocks(ncell)), dim3(256), 0, s, *p);     \
    if (p->molar) launch_wide<NEQ_, true, 1, 2>(*p, cf, cm, s);                                 \
    else launch_wide<NEQ_, false, 1, 2>(*p, cf, cm, s);                                         \
  } else {                                                                                      \
    hipLaunchKernelGGL(diff_cell_kernel<NEQ_>, dim3(blocks(ncell)), dim3(256), 0, s, *p);     \
    hipLaunchKernelGGL(diff_face_kernel<NEQ_>, dim3(blocks(nface)), dim3(256), 0, s, *p);     \
    hipLaunchKernelGGL(diff_main_kernel<NEQ_>, dim3(blocks(nint)), dim3(256), 0, s, *p);      \
  }
  switch (neq) {
    case 10: TGR_DIFF_LAUNCH(10) break;
    case 37: TGR_DIFF_LAUNCH(37) break;
    case 40: TGR_DIFF_LAUNCH(40) break;
    case 46: TGR_DIFF_LAUNCH(46) break;
    default: return -1;
  }
#undef TGR_DIFF_LAUNCH
#undef TGR_DIFF_LAUNCH2
  return hipGetLastError() == hipSuccess ? 0 : -2;
}
