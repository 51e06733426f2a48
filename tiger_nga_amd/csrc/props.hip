// Transport and equation-of-state properties on a Fortran-layout block
// (gfx950): the device restatement of
//   finitechem_W           combustion/finitechem.f90:65-74
//   finitechem_density     finitechem.f90:324-345  RHO = P_thermo W_mix / (R T)
//   finitechem_viscosity   finitechem.f90:351-411  Wilke mixing of
//                          eta_k = mucoeff_k sqrt(T) / omegamu(T kOverEps_k)
//   finitechem_diffusivity finitechem.f90:414-461  lambda from the mixture
//                          conductivities, DIFF = lambda / cp / Lewis
//   finitechem_omegamu     finitechem.f90:466-486
// over every cell of the block (ghosts included, as the reference loops over
// imino_:imaxo_ ...) whose mask is not 1.  Two mappings:
//  * props_kernel: one wavefront per cell, lane k = species k; the Wilke
//    double sum runs over j with the pair factors that depend on the molar
//    masses only, (1/sqrt 8)(1 + W_k/W_j)^-1/2 and (W_j/W_k)^1/4, precomputed
//    on the host;
//  * props_lane_kernel: one thread per cell, every lane busy in the double
//    sum.  With g_k = W_k^1/4 / sqrt(eta_k) and a_kj = (1/sqrt 8)(1 + W_k/W_j)^-1/2
//    the reference's pair term a_kj (1 + sqrt(eta_k/eta_j) (W_j/W_k)^1/4)^2 is
//    a_kj (g_k + g_j)^2 / g_k^2, so that species k's sum over j is
//      (g_k^2 sum_j a_kj y_j + 2 g_k sum_j a_kj y_j g_j + sum_j a_kj y_j g_j^2) / g_k^2:
//    three products of one constant matrix with a lane's vectors, three fused
//    multiply-adds a pair whose matrix element comes from a scalar register.
//    The diagonal a_kk = 1/4 makes j = k the reference's own term (its phi is
//    1), and with y_j = Y_j / W_j the factor W_mix cancels.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "chem_device.h"
#include "chem_kernels.h"


namespace tgr {

constexpr double kRcst = 8314.34;  // R_cst, finitechem.f90:15 (exact double)

__device__ __forceinline__ double omegamu(double t) {
  const double m1 = 3.3530622607, m2 = 2.53272006, m3 = 2.9024238575, m4 = 0.11186138893, m5 = 0.8662326188,
               m6 = 1.3913958626, m7 = 3.158490576, m8 = 0.18973411754, m9 = 0.00018682962894;
  const double num = m1 + t * (m2 + t * (m3 + t * m4));
  const double den = m5 + t * (m6 + t * (m7 + t * (m8 + t * m9)));
  return num / den;
}

// omegamu(t) as its numerator and denominator (both positive for t > 0), so
// that a caller dividing by omegamu multiplies by the denominator instead
__device__ __forceinline__ void omegamu_nd(double t, double& num, double& den) {
  const double m1 = 3.3530622607, m2 = 2.53272006, m3 = 2.9024238575, m4 = 0.11186138893, m5 = 0.8662326188,
               m6 = 1.3913958626, m7 = 3.158490576, m8 = 0.18973411754, m9 = 0.00018682962894;
  num = m1 + t * (m2 + t * (m3 + t * m4));
  den = m5 + t * (m6 + t * (m7 + t * (m8 + t * m9)));
}

template <int NEQ>
__global__ __launch_bounds__(256) void props_kernel(PropsParams p) {
  constexpr int nsp = NEQ - 1;
  constexpr TabLayout L = tab_layout<NEQ>();
  const int lane = lane_id();
  const bool sp = lane < nsp;
  const TGR_GLOBAL double* pt = (const TGR_GLOBAL double*)p.ptab;
  const double mu = sp ? pt[lane] : 0.0, koe = sp ? pt[64 + lane] : 0.0, Wk = sp ? pt[128 + lane] : 1.0;
  const double lew = (sp && p.lewis) ? p.lewis[lane] : 1.0;
  const int64_t ncell = (int64_t)p.nx * p.ny * p.nz;
  const int wpb = blockDim.x >> 6;
  for (int64_t c = (int64_t)blockIdx.x * wpb + (threadIdx.x >> 6); c < ncell; c += (int64_t)gridDim.x * wpb) {
    const int i = (int)(c % p.nx), j = (int)((c / p.nx) % p.ny), k = (int)(c / ((int64_t)p.nx * p.ny));
    if (p.mask && p.mask[p.mask_base + (int64_t)j * p.mask_ld + i] == 1) continue;
    const int64_t off = c;  // the block is the whole array
    const double Y = sp ? p.sc[(int64_t)(p.isc_sc0 + lane) * p.plane + off] : 0.0;
    const double T = p.sc[(int64_t)p.isc_T0 * p.plane + off];
    // finitechem_W: mass fractions clipped to [0, 1]
    const double yt = fmin(fmax(Y, 0.0), 1.0);
    const double Wmix = wave_sum(yt) / wave_sum(sp ? yt / Wk : 0.0);
    if (p.rho && lane == 0) p.rho[off] = p.p_thermo * Wmix / (kRcst * T);
    const double temp = fmin(fmax(T, 50.0), 5000.0);  // Tmin, Tmax (finitechem.f90:7-8)
    const double eta = sp ? mu * sqrt(temp) / omegamu(temp * koe) : 1.0;
    if (p.visc) {
      // per pair: (eta_k/eta_j)^1/2 as sqrt(eta_k) / sqrt(eta_j) and the
      // weight Y_j W_mix / W_j formed once per species (rounding-level
      // differences from the reference's expression order)
      const double se = sqrt(eta), ise = 1.0 / se, yw = sp ? Y * Wmix / Wk : 0.0;
      double sum1 = 0.0;
      for (int q = 0; q < nsp; ++q) {
        const double iseq = bcast(ise, q), ywq = bcast(yw, q);
        const double a = pt[192 + q * 64 + lane], b = pt[192 + nsp * 64 + q * 64 + lane];
        const double t1 = se * iseq * b;
        const double phi = a * ((1.0 + t1) * (1.0 + t1));
        sum1 = q != lane ? fma(ywq, phi, sum1) : sum1;
      }
      sum1 = sum1 + Y * Wmix / Wk;
      const double v = wave_sum((sp && Y > 0.0) ? (Y * Wmix * eta / (Wk * sum1)) : 0.0);
      if (lane == 0) p.visc[off] = v;
    }
    if (p.diff) {
      // COMPTHERMODATA cp at the clipped temperature (table rows in HBM)
      const TGR_GLOBAL double* th =
          (const TGR_GLOBAL double*)(p.mtab + L.th + (temp > p.tmid ? 0 : 13 * kRow)) + lane;
      const double cpk = sp ? th[448] * (th[512] + temp * (th[576] + temp * (th[640] + temp * (th[704] + temp * th[768]))))
                            : 0.0;
      const double cond = eta * (cpk + 1.25 * kRcst / Wk);
      const double s1 = wave_sum(sp ? Y * Wmix / (cond * Wk) : 0.0);
      const double s2 = wave_sum(sp ? Y * cond * Wmix / Wk : 0.0);
      const double lambda = 0.5 * (s2 + (1.0 / s1));
      const double cpm = wave_sum(Y * cpk);
      const double D = lambda / cpm;
      if (sp) p.diff[(int64_t)(p.isc_sc0 + lane) * p.plane + off] = D / lew;
      if (lane == 0) p.diff[(int64_t)p.isc_T0 * p.plane + off] = D;
      if (lane == 0 && p.isc_z0 >= 0) p.diff[(int64_t)p.isc_z0 * p.plane + off] = D;
    }
  }
}

// N doubles (even) at a wave-uniform address into scalar registers
typedef double d8 __attribute__((ext_vector_type(8), aligned(8)));
typedef double d4 __attribute__((ext_vector_type(4), aligned(8)));
typedef double d2 __attribute__((ext_vector_type(2), aligned(8)));

template <int N>
__device__ __forceinline__ void load_row(double (&m)[N], const TGR_CONST double* r) {
  constexpr int n8 = N / 8 * 8, n4 = n8 + (N - n8) / 4 * 4;
#pragma unroll
  for (int i = 0; i < n8; i += 8) {
    const d8 v = *(const TGR_CONST d8*)(r + i);
#pragma unroll
    for (int e = 0; e < 8; ++e) m[i + e] = v[e];
  }
#pragma unroll
  for (int i = n8; i < n4; i += 4) {
    const d4 v = *(const TGR_CONST d4*)(r + i);
#pragma unroll
    for (int e = 0; e < 4; ++e) m[i + e] = v[e];
  }
#pragma unroll
  for (int i = n4; i < N; i += 2) {
    const d2 v = *(const TGR_CONST d2*)(r + i);
    m[i] = v[0];
    m[i + 1] = v[1];
  }
}


// Threads of a workgroup (its g_k take 8 nsp bytes of LDS a thread, the cp rows
// 96 nsp bytes): four waves where two such workgroups fit a CU, else one, of which
// eight fit if the g_k of no more than 40 species are in LDS; EthyRedF's other
// five are in registers.  Workgroups of two waves with all g_k in LDS leave EthyRedF
// six waves a CU and a second, nearly empty round from 98,305 cells: 100,000 /
// 131,072 / 1,000,000 cells 130 / 140 / 695 us, this way 80 / 83 / 638; DME39, 50,000
// / 262,144 cells: 59 / 180 us with two waves, 54 / 147 with four, 51 / 133 with one.
// The cp rows are in LDS where they do not cost a resident workgroup.
constexpr int kLdsBytes = 160 * 1024;
template <int NEQ>
constexpr int props_block() {
  return 2 * (256 * 8 + 96) * (NEQ - 1) <= kLdsBytes ? 256 : 64;
}
template <int NEQ>
constexpr int props_lds_species() {
  const int fit = kLdsBytes / 8 / (props_block<NEQ>() * 8);
  return props_block<NEQ>() == 64 && NEQ - 1 > fit ? fit : NEQ - 1;
}
template <int NEQ>
constexpr bool props_cp_lds() {
  return kLdsBytes / ((props_block<NEQ>() * 8 + 96) * (NEQ - 1)) == kLdsBytes / (props_block<NEQ>() * 8 * (NEQ - 1));
}

// One thread per cell (the block's cells in their storage order, so every
// field access is coalesced).  A first loop over the species forms W_mix, the
// conductivity sums and g (to LDS; in registers for up to 20 species); then, for
// a part of the species k at a time, a loop over j adds column j of the pair
// matrix times y_j, y_j g_j and y_j g_j^2 to the part's sums: 3 x 18 independent
// chains (GRI-3.0), the next column's scalar loads under way.  Bound by VALU
// issue (64 % busy, 8,400 instructions a wave of which 3,900 are the pairs');
// 130^3 GRI-3.0 cells in 0.83 ms, 1.03 ms with a 16-byte LDS read per pair.  Sums
// run in species order (the wave kernel's are tree reductions) and eta = mucoeff sqrt(T) den / num takes
// omegamu's numerator and denominator with one division: rounding-level
// differences.
template <int NEQ>
__global__ __launch_bounds__(props_block<NEQ>()) __attribute__((amdgpu_waves_per_eu(2))) void props_lane_kernel(
    PropsParams p) {
  constexpr int nsp = NEQ - 1, kBlock = props_block<NEQ>(), kPart = kPropsPart(nsp);
  constexpr TabLayout L = tab_layout<NEQ>();
  constexpr int kPair = 192 + 2 * nsp * 64;
  constexpr bool kOne = kPropsParts(nsp) == 1;  // few species: one part, everything in registers
  // g_k of kLds species in LDS, of the kReg past them in registers
  constexpr int kLds = kOne ? 1 : props_lds_species<NEQ>(), kReg = kOne ? 0 : nsp - kLds;
  __shared__ double gs[kLds][kBlock];
  double gr[kReg ? kReg : 1];
  constexpr bool kCpLds = props_cp_lds<NEQ>();
  __shared__ __attribute__((aligned(16))) double cps[kCpLds ? nsp * 12 : 2];  // cp rows, [species][T > tmid][6]
  if constexpr (kCpLds) {
    for (int t = threadIdx.x; t < nsp * 12; t += kBlock) {
      const int k = t / 12, hi = (t / 6) % 2, c = t % 6;
      cps[t] = *(const double*)(p.mtab + L.th + (hi ? 0 : 13 * kRow) + (7 + c) * kRow + k * 8);
    }
    __syncthreads();
  }
  const int64_t ncell = (int64_t)p.nx * p.ny * p.nz;
  const int64_t c = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (c >= ncell) return;
  if (p.mask && p.mask[p.mask_base + (int64_t)((c / p.nx) % p.ny) * p.mask_ld + (int)(c % p.nx)] == 1) return;
  const TGR_CONST double* pt = (const TGR_CONST double*)p.ptab;
  const TGR_CONST double* w14 = pt + kPair + nsp * kPropsParts(nsp) * kPart;
  const TGR_CONST double* w12 = w14 + nsp;
  const TGR_GLOBAL double* ys = (const TGR_GLOBAL double*)p.sc + (int64_t)p.isc_sc0 * p.plane + c;
  const double T = p.sc[(int64_t)p.isc_T0 * p.plane + c];
  const TGR_CONST double* iw = (const TGR_CONST double*)(p.mtab + L.iw);  // 1 / W_k
  const double temp = fmin(fmax(T, 50.0), 5000.0);  // Tmin, Tmax (finitechem.f90:7-8)
  const double st = sqrt(temp);
  const bool hi = temp > p.tmid;
  const double* cr = cps + (hi ? 6 : 0);
  const TGR_CONST double* thi = (const TGR_CONST double*)(p.mtab + L.th);
  const TGR_CONST double* tlo = thi + 13 * 64;
  // Both loops take kCh species at a time: the next chunk's Y are loaded while
  // one computes (a load takes longer than one species), and the chains of a
  // chunk's species overlap.
  constexpr int kCh = kOne ? nsp : (kReg ? kReg : 4);
  constexpr int kLoop = kReg ? kLds : nsp;  // species of the loops; the ones in registers are one chunk more
  static_assert(!kReg || kLds % kCh == 0, "whole chunks");
  double Yn[kCh];
#pragma unroll
  for (int u = 0; u < kCh; ++u) Yn[u] = ys[(u < nsp ? u : 0) * p.plane];
  // finitechem_W: mass fractions clipped to [0, 1]
  double sy = 0.0, syw = 0.0, s1 = 0.0, s2 = 0.0, cpm = 0.0;
  double g1[kOne ? nsp : 1];
#pragma unroll
  for (int tail = 0; tail < (kReg ? 2 : 1); ++tail)
#pragma unroll 1  // (one turn of the tail: its register indices are constants)
  for (int k0 = tail ? kLds : 0; k0 < (tail ? nsp : kLoop); k0 += kCh) {
    double Yc[kCh];
#pragma unroll
    for (int u = 0; u < kCh; ++u) {
      const int kn = k0 + kCh + u;
      Yc[u] = Yn[u];
      if constexpr (kCh < nsp) Yn[u] = ys[(kn < nsp ? kn : 0) * p.plane];
    }
#pragma unroll
    for (int u = 0; u < kCh; ++u) {
      const int k = k0 + u;
      if (nsp % kCh && k >= nsp) break;
      const double Y = Yc[u];
      const double yt = fmin(fmax(Y, 0.0), 1.0);
      sy += yt;
      syw = fma(yt, iw[k], syw);
      double num, den;
      omegamu_nd(temp * pt[64 + k], num, den);
      const double ms = pt[k] * st * den;
      if (p.visc) {
        const double g = w14[k] * sqrt(num / ms);
        if constexpr (kOne) g1[u] = g;
        else if (tail) gr[k - kLds] = g;
        else gs[k][threadIdx.x] = g;
      }
      if (p.diff) {
        const double eta = ms / num;
        double d[6];
#pragma unroll
        for (int e = 0; e < 6; ++e) {
          if constexpr (kCpLds) d[e] = cr[k * 12 + e];
          else d[e] = hi ? thi[(7 + e) * 64 + k] : tlo[(7 + e) * 64 + k];
        }
        const double cpk = d[0] * (d[1] + temp * (d[2] + temp * (d[3] + temp * (d[4] + temp * d[5]))));
        const double cond = eta * fma(1.25 * kRcst, iw[k], cpk);
        const double yk = Y * iw[k];
        s1 += yk / cond;
        s2 += yk * cond;
        cpm += Y * cpk;
      }
    }
  }
  const double Wmix = sy / syw;
  if (p.rho) p.rho[c] = p.p_thermo * Wmix / (kRcst * T);
  if (p.visc) {
    double visc = 0.0;
    if constexpr (kOne) {
      const TGR_CONST double* col = pt + kPair;
#pragma unroll
      for (int k = 0; k < nsp; ++k) {
        double a = 0.0, b = 0.0, d = 0.0;
#pragma unroll
        for (int q = 0; q < nsp; ++q) {
          const double y = Yn[q] * iw[q], yg = y * g1[q];
          a = fma(col[q * kPart + k], y, a);
          b = fma(col[q * kPart + k], yg, b);
          d = fma(col[q * kPart + k], yg * g1[q], d);
        }
        const double s = fma(g1[k], fma(g1[k], a, 2.0 * b), d);
        visc += Yn[k] > 0.0 ? Yn[k] * iw[k] * w12[k] / s : 0.0;
      }
    }
#pragma unroll
    for (int k0 = 0; k0 < (kOne ? 0 : nsp); k0 += kPart) {
      const TGR_CONST double* col = pt + kPair + (k0 / kPart) * nsp * kPart;  // [part][j][kPart]
      double a[kPart], b[kPart], d[kPart], m[kPart];
#pragma unroll
      for (int k = 0; k < kPart; ++k) a[k] = b[k] = d[k] = 0.0;
      load_row(m, col);
#pragma unroll
      for (int u = 0; u < kCh; ++u) Yn[u] = ys[(u < nsp ? u : 0) * p.plane];
#pragma unroll
      for (int tail = 0; tail < (kReg ? 2 : 1); ++tail)
#pragma unroll 1
      for (int q0 = tail ? kLds : 0; q0 < (tail ? nsp : kLoop); q0 += kCh) {
        double Yc[kCh];
#pragma unroll
        for (int u = 0; u < kCh; ++u) {
          const int qn = q0 + kCh + u;
          Yc[u] = Yn[u];
          if constexpr (kCh < nsp) Yn[u] = ys[(qn < nsp ? qn : 0) * p.plane];
        }
#pragma unroll
        for (int u = 0; u < kCh; ++u) {
          const int q = q0 + u;
          if (nsp % kCh && q >= nsp) break;
          double mn[kPart];
          load_row(mn, col + (q + 1 < nsp ? q + 1 : 0) * kPart);
          double g;
          if (tail) g = gr[q - kLds];
          else g = gs[q][threadIdx.x];
          const double y = Yc[u] * iw[q], yg = y * g, ygg = yg * g;
#pragma unroll
          for (int k = 0; k < kPart; ++k) {
            a[k] = fma(m[k], y, a[k]);
            b[k] = fma(m[k], yg, b[k]);
            d[k] = fma(m[k], ygg, d[k]);
          }
#pragma unroll
          for (int k = 0; k < kPart; ++k) m[k] = mn[k];
        }
      }
#pragma unroll
      for (int k = 0; k < kPart; ++k)
        if (k0 + k < nsp) {
          const double Y = ys[(k0 + k) * p.plane], g = k0 + k < kLds ? gs[k0 + k < kLds ? k0 + k : 0][threadIdx.x]
                                                                          : gr[k0 + k < kLds ? 0 : k0 + k - kLds];
          const double s = fma(g, fma(g, a[k], 2.0 * b[k]), d[k]);
          visc += Y > 0.0 ? Y * iw[k0 + k] * w12[k0 + k] / s : 0.0;
        }
    }
    p.visc[c] = visc;
  }
  if (p.diff) {
    const double D = 0.5 * (s2 * Wmix + (1.0 / (s1 * Wmix))) / cpm;
#pragma unroll 1
    for (int k = 0; k < nsp; ++k) p.diff[(int64_t)(p.isc_sc0 + k) * p.plane + c] = p.lewis ? D / p.lewis[k] : D;
    p.diff[(int64_t)p.isc_T0 * p.plane + c] = D;
    if (p.isc_z0 >= 0) p.diff[(int64_t)p.isc_z0 * p.plane + c] = D;
  }
}

}  // namespace tgr

using namespace tgr;

extern "C" int tgr_launch_props(const PropsParams* p, int neq, int lane_map, hipStream_t s) {
  const int64_t ncell = (int64_t)p->nx * p->ny * p->nz;
  if (ncell <= 0) return 0;
  if (lane_map) {
#define TGR_PROPS_LAUNCH(NEQ_)                                                                                   \
  case NEQ_: {                                                                                                  \
    const int64_t nb = (ncell + props_block<NEQ_>() - 1) / props_block<NEQ_>();                                 \
    if (nb > 0x7fffffff) return -1;                                                                             \
    hipLaunchKernelGGL(props_lane_kernel<NEQ_>, dim3((unsigned)nb), dim3(props_block<NEQ_>()), 0, s, *p);       \
    break;                                                                                                      \
  }
    switch (neq) {
      TGR_PROPS_LAUNCH(10)
      TGR_PROPS_LAUNCH(37)
      TGR_PROPS_LAUNCH(40)
      TGR_PROPS_LAUNCH(46)
      default: return -1;
    }
#undef TGR_PROPS_LAUNCH
    return hipGetLastError() == hipSuccess ? 0 : -2;
  }
  const int64_t need = (ncell + 3) / 4;
  const dim3 grid((unsigned)(need < 8192 ? need : 8192)), block(256);
  switch (neq) {
    case 10: hipLaunchKernelGGL(props_kernel<10>, grid, block, 0, s, *p); break;
    case 37: hipLaunchKernelGGL(props_kernel<37>, grid, block, 0, s, *p); break;
    case 40: hipLaunchKernelGGL(props_kernel<40>, grid, block, 0, s, *p); break;
    case 46: hipLaunchKernelGGL(props_kernel<46>, grid, block, 0, s, *p); break;
    default: return -1;
  }
  return hipGetLastError() == hipSuccess ? 0 : -2;
}
