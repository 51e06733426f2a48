/* Generated by tiger_nga_amd/mech/lanegen.py from the compiled mechanism h2
 * (reference combustion/HYDROGENF.f90).  Do not edit.  Lane-per-state right-hand side of
 * finitechem_compute_rhs (combustion/finitechem.f90:93-175). */
#pragma once
#include "lane_rhs.h"

namespace tgr {

template <>
struct LaneRhs<10> {
  // production rates cd (kmol/m3/s) from the concentrations, temperature and pressure of this lane's state
  static __device__ __forceinline__ void rates(const double (&C)[9], double T, double P, double (&cd)[9]) {
    const double C0 = C[0];
    const double C1 = C[1];
    const double C2 = C[2];
    const double C3 = C[3];
    const double C4 = C[4];
    const double C5 = C[5];
    const double C6 = C[6];
    const double C7 = C[7];
    const double C8 = C[8];
    const double lt = flog2(T * (1.0 / kTUnit));
    const double rt = kRgasF4 * T;
    const double irt = kLog2e / rt;
    const double invT = 1.0 / T;
    const double p_rt = P / rt;
    double ctot = C0;
    ctot += C1;
    ctot += C2;
    ctot += C3;
    ctot += C4;
    ctot += C5;
    ctot += C6;
    ctot += C7;
    ctot += C8;
    auto M0 = [&]() { double s_ = ctot; s_ = fma(-0x1.0000000000000p+0, C5, s_); s_ = fma(-0x1.0000000000000p+0, C6, s_); return s_; };
    auto M1 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.5333340000000p+2, C6, s_); return s_; };
    auto M2 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.6000000000000p+3, C6, s_); return s_; };
    auto M3 = [&]() { double s_ = ctot; s_ = fma(0x1.6666680000000p+0, C5, s_); s_ = fma(0x1.cccccc0000000p+3, C6, s_); return s_; };
    auto M4 = [&]() { double s_ = ctot; s_ = fma(-0x1.3333300000000p-3, C2, s_); s_ = fma(-0x1.0000000000000p-2, C5, s_); s_ = fma(0x1.5c7ae20000000p+3, C6, s_); return s_; };
    double cd0 = 0.0;
    double cd1 = 0.0;
    double cd2 = 0.0;
    double cd3 = 0.0;
    double cd4 = 0.0;
    double cd5 = 0.0;
    double cd6 = 0.0;
    double cd7 = 0.0;
    double cd8 = 0.0;
    {  // R1 (elementary)
    const double kf = 0x1.7843b02d8edbcp+38 * fexp2(fma(-0x1.0ffce80000000p+26, irt, -0x1.570a3e0000000p-1 * lt));
    const double kb = 0x1.6ca1517eac207p+33 * fexp2(fma(-0x1.d45d120000000p+18, irt, -0x1.dfd3f60000000p-3 * lt));
    const double q = kf * C1 * C2 - kb * C4 * C3;
    cd1 -= q;
    cd2 -= q;
    cd3 += q;
    cd4 += q;
    }
    {  // R2 (elementary)
    const double kf = 0x1.c4138c8783e65p+29 * fexp2(fma(-0x1.8fa0b00000000p+24, irt, 0x1.59999a0000000p+1 * lt));
    const double kb = 0x1.b09beee7aedabp+28 * fexp2(fma(-0x1.32b5e60000000p+24, irt, 0x1.54f90a0000000p+1 * lt));
    const double q = kf * C3 * C5 - kb * C4 * C1;
    cd1 += q;
    cd3 -= q;
    cd4 += q;
    cd5 -= q;
    }
    {  // R3 (elementary)
    const double kf = 0x1.fc9bd5fddb67fp+30 * fexp2(fma(-0x1.b5ed600000000p+23, irt, 0x1.828f5c0000000p+0 * lt));
    const double kb = 0x1.6e268e0975208p+33 * fexp2(fma(-0x1.273c980000000p+26, irt, 0x1.6800000000000p+0 * lt));
    const double q = kf * C4 * C5 - kb * C6 * C1;
    cd1 += q;
    cd4 -= q;
    cd5 -= q;
    cd6 += q;
    }
    {  // R4 (elementary)
    const double kf = 0x1.e1645174bab52p+26 * fexp2(fma(0x1.0d78600000000p+23, irt, 0x1.3333340000000p+1 * lt));
    const double kb = 0x1.6a2cb0cfb1368p+30 * fexp2(fma(-0x1.cc15240000000p+25, irt, 0x1.2a8c6a0000000p+1 * lt));
    const double q = kf * C4 * C4 - kb * C6 * C3;
    cd3 += q;
    cd4 = fma(-0x1.0000000000000p+1, q, cd4);
    cd6 += q;
    }
    {  // R6 (elementary)
    const double kf = 0x1.fc2efa228911cp+30 * fexp2(fma(0.0, irt, -0x1.3333340000000p-1 * lt));
    const double kb = 0x1.01c987be36767p+42 * fexp2(fma(-0x1.9d073a0000000p+28, irt, -0x1.ff84ca0000000p-3 * lt));
    const double q = kf * C1 * C1 * C5 - kb * C5 * C5;
    cd1 = fma(-0x1.0000000000000p+1, q, cd1);
    cd5 += q;
    }
    {  // R7 (elementary)
    const double kf = 0x1.57d996ec49561p+34 * fexp2(fma(0.0, irt, -0x1.4000000000000p+0 * lt));
    const double kb = 0x1.5cd9cbf288374p+45 * fexp2(fma(-0x1.9d073a0000000p+28, irt, -0x1.ccae000000000p-1 * lt));
    const double q = kf * C1 * C1 * C6 - kb * C6 * C5;
    cd1 = fma(-0x1.0000000000000p+1, q, cd1);
    cd5 += q;
    }
    {  // R13 (elementary)
    const double kf = 0x1.0e7e8553d6572p+31 * fexp2(fma(-0x1.aaf5c20000000p+27, irt, 0x1.370a3e0000000p+1 * lt));
    const double kb = 0x1.5c5e5c4537e01p+30 * fexp2(fma(0x1.1727a20000000p+22, irt, 0x1.08b1ee0000000p+1 * lt));
    const double q = kf * C5 * C2 - kb * C1 * C7;
    cd1 += q;
    cd2 -= q;
    cd5 -= q;
    cd7 += q;
    }
    {  // R15 (elementary)
    const double kf = 0x1.d942c90000000p+31 * fexp2(fma(-0x1.5704800000000p+21, irt, 0.0 * lt));
    const double kb = 0x1.005fb2a02b18ep+30 * fexp2(fma(-0x1.aa36420000000p+27, irt, 0x1.6358b00000000p-1 * lt));
    const double q = kf * C7 * C1 - kb * C6 * C3;
    cd1 -= q;
    cd3 += q;
    cd6 += q;
    cd7 -= q;
    }
    {  // R16 (elementary)
    const double kf = 0x1.170634d000000p+36 * fexp2(fma(-0x1.44b5000000000p+21, irt, 0.0 * lt));
    const double kb = 0x1.91d3c5155ebcdp+30 * fexp2(fma(-0x1.2610340000000p+27, irt, 0x1.85f4800000000p-1 * lt));
    const double q = kf * C7 * C1 - kb * C4 * C4;
    cd1 -= q;
    cd4 = fma(0x1.0000000000000p+1, q, cd4);
    cd7 -= q;
    }
    {  // R17 (elementary)
    const double kf = 0x1.2a05f20000000p+35 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.bae11a0ddf410p+34 * fexp2(fma(-0x1.a811a60000000p+27, irt, 0x1.4dbe3c0000000p-2 * lt));
    const double q = kf * C7 * C3 - kb * C2 * C4;
    cd2 += q;
    cd3 -= q;
    cd4 += q;
    cd7 -= q;
    }
    {  // R18 (elementary)
    const double kf = 0x1.62a5cb8000000p+34 * fexp2(fma(0x1.fe41000000000p+20, irt, 0.0 * lt));
    const double kb = 0x1.8c7f6cffb4e41p+37 * fexp2(fma(-0x1.13f8fa0000000p+28, irt, 0x1.0886e00000000p-2 * lt));
    const double q = kf * C7 * C4 - kb * C2 * C6;
    cd2 += q;
    cd4 -= q;
    cd6 += q;
    cd7 -= q;
    }
    {  // R19 (elementary)
    const double kf = 0x1.2309ce5400000p+43 * fexp2(fma(-0x1.149a8c0000000p+26, irt, 0.0 * lt));
    const double kb = 0x1.4561d91d0b10ap+46 * fexp2(fma(-0x1.5b1dde0000000p+28, irt, 0x1.0886e00000000p-2 * lt));
    const double q = kf * C7 * C4 - kb * C2 * C6;
    cd2 += q;
    cd4 -= q;
    cd6 += q;
    cd7 -= q;
    }
    {  // R20 (elementary)
    const double kf = 0x1.efe9200000000p+26 * fexp2(fma(0x1.a042800000000p+22, irt, 0.0 * lt));
    const double kb = 0x1.41dc57b6679e3p+30 * fexp2(fma(-0x1.27309e2000000p+27, irt, -0x1.f587500000000p-3 * lt));
    const double q = kf * C7 * C7 - kb * C8 * C2;
    cd2 += q;
    cd7 = fma(-0x1.0000000000000p+1, q, cd7);
    cd8 += q;
    }
    {  // R21 (elementary)
    const double kf = 0x1.54dd333000000p+38 * fexp2(fma(-0x1.7f12680000000p+25, irt, 0.0 * lt));
    const double kb = 0x1.ba76366cf4b52p+41 * fexp2(fma(-0x1.93f74c2000000p+27, irt, -0x1.f587500000000p-3 * lt));
    const double q = kf * C7 * C7 - kb * C8 * C2;
    cd2 += q;
    cd7 = fma(-0x1.0000000000000p+1, q, cd7);
    cd8 += q;
    }
    {  // R22 (elementary)
    const double kf = 0x1.7a20000000000p+30 * fexp2(fma(-0x1.4c08000000000p+24, irt, 0x1.0000000000000p+1 * lt));
    const double kb = 0x1.c45fd1fbb8faep+27 * fexp2(fma(-0x1.51fa9a0000000p+26, irt, 0x1.4db0de0000000p+1 * lt));
    const double q = kf * C8 * C1 - kb * C5 * C7;
    cd1 -= q;
    cd5 += q;
    cd7 += q;
    cd8 -= q;
    }
    {  // R23 (elementary)
    const double kf = 0x1.671e344000000p+34 * fexp2(fma(-0x1.fae5a00000000p+23, irt, 0.0 * lt));
    const double kb = 0x1.bd6ba1d6bdd74p+28 * fexp2(fma(-0x1.1c33be0000000p+28, irt, 0x1.43cc8e0000000p+0 * lt));
    const double q = kf * C8 * C1 - kb * C4 * C6;
    cd1 -= q;
    cd4 += q;
    cd6 += q;
    cd8 -= q;
    }
    {  // R24 (elementary)
    const double kf = 0x1.2cf0000000000p+31 * fexp2(fma(-0x1.fae5a00000000p+23, irt, 0x1.0000000000000p+1 * lt));
    const double kb = 0x1.5886cc65ad2cfp+27 * fexp2(fma(-0x1.271a9c0000000p+26, irt, 0x1.49104e0000000p+1 * lt));
    const double q = kf * C8 * C3 - kb * C4 * C7;
    cd3 -= q;
    cd4 += q;
    cd7 += q;
    cd8 -= q;
    }
    {  // R25 (elementary)
    const double kf = 0x1.dcd6500000000p+30 * fexp2(fma(-0x1.b503000000000p+20, irt, 0.0 * lt));
    const double kb = 0x1.9ab1df792d772p+30 * fexp2(fma(-0x1.f64b920000000p+26, irt, 0x1.01a5440000000p-1 * lt));
    const double q = kf * C8 * C4 - kb * C6 * C7;
    cd4 -= q;
    cd6 += q;
    cd7 += q;
    cd8 -= q;
    }
    {  // R26 (elementary)
    const double kf = 0x1.91bca8b63554cp+64 * fexp2(fma(-0x1.2c10680000000p+27, irt, -0x1.c000000000000p+2 * lt));
    const double kb = 0x1.5a00d8b7b4582p+64 * fexp2(fma(-0x1.11e6160000000p+28, irt, -0x1.9fcb680000000p+2 * lt));
    const double q = kf * C8 * C4 - kb * C6 * C7;
    cd4 -= q;
    cd6 += q;
    cd7 += q;
    cd8 -= q;
    }
    {  // R5 (third_body)
    const double kf = 0x1.9e70448800000p+31 * fexp2(fma(0.0, irt, -0x1.0000000000000p+0 * lt));
    const double kb = 0x1.a4774983c45ebp+42 * fexp2(fma(-0x1.9d073a0000000p+28, irt, -0x1.4cae000000000p-1 * lt));
    const double q = (kf * C1 * C1 - kb * C5) * M0();
    cd1 = fma(-0x1.0000000000000p+1, q, cd1);
    cd5 += q;
    }
    {  // R9 (third_body)
    const double kf = 0x1.38a388a43c000p+37 * fexp2(fma(0.0, irt, -0x1.0000000000000p+1 * lt));
    const double kb = 0x1.c8b3c265a295cp+50 * fexp2(fma(-0x1.d926f40000000p+28, irt, -0x1.c0e6080000000p+0 * lt));
    const double q = (kf * C1 * C4 - kb * C6) * M1();
    cd1 -= q;
    cd4 -= q;
    cd6 += q;
    }
    {  // R10 (third_body)
    const double kf = 0x1.1272f99b80000p+34 * fexp2(fma(0.0, irt, -0x1.0000000000000p+0 * lt));
    const double kb = 0x1.0a72723925450p+44 * fexp2(fma(-0x1.97388e0000000p+28, irt, -0x1.5f30840000000p-1 * lt));
    const double q = (kf * C1 * C3 - kb * C4) * M2();
    cd1 -= q;
    cd3 -= q;
    cd4 += q;
    }
    {  // R14 (falloff)
    const double kinf_f = 0x1.48f5c74fe0810p+33 * fexp2(fma(0.0, irt, -0x1.7ae1480000000p-2 * lt));
    const double k0_f = 0x1.417095c517ea1p+32 * fexp2(fma(0x1.24a9e00000000p+23, irt, -0x1.28f5c20000000p-1 * lt));
    const double kinf_b = 0x1.836985586c056p+52 * fexp2(fma(-0x1.9994c60000000p+27, irt, -0x1.636b900000000p+0 * lt));
    const double k0_b = 0x1.7a8e47c96d4d4p+51 * fexp2(fma(-0x1.874a280000000p+27, irt, -0x1.992e1e0000000p+0 * lt));
    const double m_ = M2();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.0fc5040000000p-2, fexp2(-(0x1.f6ead796c4570p-7 * T)), fc);
    fc = fma(0x1.781d7e0000000p-1, fexp2(-(0x1.aebea4d2c5521p-11 * T)), fc);
    fc = fma(0x1.0000000000000p+0, fexp2(-(0x1.d340bb31e6c59p+12 * invT)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C4 * C4 - kb * C8;
    cd4 = fma(-0x1.0000000000000p+1, q, cd4);
    cd8 += q;
    }
    {  // R11 (third_body)
    const double kf = 0x1.bf08eb0000000p+27 * fexp2(fma(0.0, irt, -0x1.0000000000000p+0 * lt));
    const double kb = 0x1.bfd6620e8f8eap+42 * fexp2(fma(-0x1.dac2b02000000p+28, irt, -0x1.1f23240000000p+0 * lt));
    const double q = (kf * C3 * C3 - kb * C2) * M3();
    cd2 += q;
    cd3 = fma(-0x1.0000000000000p+1, q, cd3);
    }
    {  // R12 (falloff)
    const double kinf_f = 0x1.28d4aaa8ae8d5p+36 * fexp2(fma(0.0, irt, 0x1.c28f5c0000000p-2 * lt));
    const double k0_f = 0x1.2fdc9732a2fe5p+33 * fexp2(fma(0.0, irt, -0x1.6666660000000p+0 * lt));
    const double kinf_b = 0x1.83d671c7e1accp+46 * fexp2(fma(-0x1.865f740000000p+27, irt, 0x1.b66fd60000000p-2 * lt));
    const double k0_b = 0x1.8d0597e44972ep+43 * fexp2(fma(-0x1.865f740000000p+27, irt, -0x1.696e580000000p+0 * lt));
    const double m_ = M4();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.0000000000000p-1, fexp2(-(0x1.235995d2649cap+100 * T)), fc);
    fc = fma(0x1.0000000000000p-1, fexp2(-(0x1.d42e69bdf23bep-100 * T)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C1 * C2 - kb * C7;
    cd1 -= q;
    cd2 -= q;
    cd7 += q;
    }
    cd[0] = cd0;
    cd[1] = cd1;
    cd[2] = cd2;
    cd[3] = cd3;
    cd[4] = cd4;
    cd[5] = cd5;
    cd[6] = cd6;
    cd[7] = cd7;
    cd[8] = cd8;
  }

  // s: [rho*Y (9), rho*T] of this lane's state; f: the right-hand side
  static __device__ __forceinline__ void eval(const double (&s)[10], double P, double (&f)[10]) {
    double rho = s[0];
    rho += s[1];
    rho += s[2];
    rho += s[3];
    rho += s[4];
    rho += s[5];
    rho += s[6];
    rho += s[7];
    rho += s[8];
    const double T = s[9] / rho;
    const double irho = 1.0 / rho;
    double C[9], cd[9];
    C[0] = s[0] * 0x1.245cd2eb40a46p-5;
    C[1] = s[1] * 0x1.fbefbe72dfd0bp-1;
    C[2] = s[2] * 0x1.0000000000000p-5;
    C[3] = s[3] * 0x1.0000000000000p-4;
    C[4] = s[4] * 0x1.e1a7dc7865ca7p-5;
    C[5] = s[5] * 0x1.fbefbe72dfd0bp-2;
    C[6] = s[6] * 0x1.c6b4f7f1539dfp-5;
    C[7] = s[7] * 0x1.f05d519a5a4afp-6;
    C[8] = s[8] * 0x1.e1a7dc7865ca7p-6;
    const bool hi = T > 0x1.f400000000000p+9;
    double cpm = 0.0;
    if (hi) {
      cpm = fma(s[0] * irho, 0x1.28ba9057d1783p+8 * (0x1.769c23b7952d2p+1 + T * (0x1.86106ec5d7fc6p-10 + T * (-0x1.3132bf1b89c39p-21 + T * (0x1.bc128a9b8a724p-34 + T * -0x1.e6a15668d1fd9p-48)))), cpm);
      cpm = fma(s[1] * irho, 0x1.01c2d34acaff7p+13 * (0x1.40000015798eep+1 + T * (-0x1.961a6ec6a1e45p-36 + T * (0x1.230b4c341c642p-46 + T * (-0x1.5d647fbe2e672p-58 + T * 0x1.2d244e9510ba2p-71)))), cpm);
      cpm = fma(s[2] * irho, 0x1.03d2b851eb852p+8 * (0x1.a42a332f575b8p+1 + T * (0x1.84c851ecf574dp-10 + T * (-0x1.96ee255022a3dp-21 + T * (0x1.cca1706e20348p-33 + T * -0x1.8667712a69c18p-46)))), cpm);
      cpm = fma(s[3] * irho, 0x1.03d2b851eb852p+9 * (0x1.48e2c7b5e1a3dp+1 + T * (-0x1.689a006cdb509p-14 + T * (0x1.6855a2fbdda5cp-25 + T * (-0x1.607823c010ceap-37 + T * 0x1.620b4436bd152p-50)))), cpm);
      cpm = fma(s[4] * irho, 0x1.e8d949731098dp+8 * (0x1.6eaf6f6ecdbe1p+1 + T * (0x1.14f4d0c23ad0ap-10 + T * (-0x1.163020518c34ep-22 + T * (0x1.0c7922a4a2d04p-35 + T * -0x1.7fe9359e80e81p-50)))), cpm);
      cpm = fma(s[5] * irho, 0x1.01c2d350092cdp+12 * (0x1.ab2bf6fecf7e5p+1 + T * (-0x1.9e6b00cea2ba4p-15 + T * (0x1.0c24d11e93b22p-21 + T * (-0x1.8adee4a4b6baep-33 + T * 0x1.68bf7de4136dcp-46)))), cpm);
      cpm = fma(s[6] * irho, 0x1.cd7f5ff609dd0p+8 * (0x1.8459ddac6e07ap+1 + T * (0x1.1d553f9364039p-9 + T * (-0x1.6057d217698d4p-23 + T * (-0x1.aacb906a5f7ccp-34 + T * 0x1.2f01042cd6ffep-46)))), cpm);
      cpm = fma(s[7] * irho, 0x1.f7c6fae7924afp+7 * (0x1.0119fbbf289f6p+2 + T * (0x1.2593e46a1f9dfp-9 + T * (-0x1.5431502070c84p-21 + T * (0x1.f675fa32f618cp-34 + T * -0x1.84c80e71ea191p-47)))), cpm);
      cpm = fma(s[8] * irho, 0x1.e8d94983d7907p+7 * (0x1.0a8f681d1fcb7p+2 + T * (0x1.41abe4bc5704bp-8 + T * (-0x1.fe66ae3495cc5p-20 + T * (0x1.981f91177d524p-32 + T * -0x1.0353229ef325dp-45)))), cpm);
    } else {
      cpm = fma(s[0] * irho, 0x1.28ba9057d1783p+8 * (0x1.a63b0c4588a05p+1 + T * (0x1.712969da04050p-10 + T * (-0x1.09f7a2b098bd4p-18 + T * (0x1.83ae94da0fe59p-28 + T * -0x1.581526048e0d6p-39)))), cpm);
      cpm = fma(s[1] * irho, 0x1.01c2d34acaff7p+13 * (0x1.4000000000000p+1 + T * (0x1.8d112bff6d580p-41 + T * (-0x1.1fa470055807fp-49 + T * (0x1.538a620b2373fp-59 + T * -0x1.1863cffe0b329p-70)))), cpm);
      cpm = fma(s[2] * irho, 0x1.03d2b851eb852p+8 * (0x1.e42787ae5fa45p+1 + T * (-0x1.88c9b66c8c0dfp-9 + T * (0x1.4a6bae1fdae75p-17 + T * (-0x1.4ca5927ada53cp-27 + T * 0x1.c883a18b02bcdp-39)))), cpm);
      cpm = fma(s[3] * irho, 0x1.03d2b851eb852p+9 * (0x1.9589c6bdbf12dp+1 + T * (-0x1.add3ae5787a18p-9 + T * (0x1.bdcef845b6ae0p-18 + T * (-0x1.a51e14d5c0503p-28 + T * 0x1.2954967e1b470p-39)))), cpm);
      cpm = fma(s[4] * irho, 0x1.e8d949731098dp+8 * (0x1.080501d23d242p+2 + T * (-0x1.a6c41f4a374cap-9 + T * (0x1.b6101eb7dedbep-18 + T * (-0x1.8e78ee8164a9cp-28 + T * 0x1.2240d8be85bd5p-39)))), cpm);
      cpm = fma(s[5] * irho, 0x1.01c2d350092cdp+12 * (0x1.2c130ac9b2911p+1 + T * (0x1.058175d02a941p-7 + T * (-0x1.46ca05831775cp-16 + T * (0x1.5a4c582f87e3dp-26 + T * -0x1.03862939e564dp-37)))), cpm);
      cpm = fma(s[6] * irho, 0x1.cd7f5ff609dd0p+8 * (0x1.0cb686e536fbfp+2 + T * (-0x1.0aeb63b84c925p-9 + T * (0x1.b593a7c039b70p-18 + T * (-0x1.7921667072d59p-28 + T * 0x1.f2c47bce627b1p-40)))), cpm);
      cpm = fma(s[7] * irho, 0x1.f7c6fae7924afp+7 * (0x1.1350a899bcaa1p+2 + T * (-0x1.373d054674594p-8 + T * (0x1.62fa28e3a8ea6p-16 + T * (-0x1.a110b0905e0fcp-26 + T * 0x1.46f1288fc5c1cp-37)))), cpm);
      cpm = fma(s[8] * irho, 0x1.e8d94983d7907p+7 * (0x1.11abd48f63e0ap+2 + T * (-0x1.1c98643a78c6ap-11 + T * (0x1.18be22e62f026p-16 + T * (-0x1.72b101d35ae59p-26 + T * 0x1.2f72fba30b7c2p-37)))), cpm);
    }
    rates(C, T, P, cd);
    f[0] = cd[0] * 0x1.c051ec0000000p+4;
    f[1] = cd[1] * 0x1.020c4a0000000p+0;
    f[2] = cd[2] * 0x1.0000000000000p+5;
    f[3] = cd[3] * 0x1.0000000000000p+4;
    f[4] = cd[4] * 0x1.1020c40000000p+4;
    f[5] = cd[5] * 0x1.020c4a0000000p+1;
    f[6] = cd[6] * 0x1.20418a0000000p+4;
    f[7] = cd[7] * 0x1.0810620000000p+5;
    f[8] = cd[8] * 0x1.1020c40000000p+5;
    double tmp = 0.0;
    if (hi) {
      tmp = fma(-(0x1.28ba9057d1783p+8 * (T * (0x1.769c23b7952d2p+1 + T * (0x1.86106ec5d7fc6p-11 + T * (-0x1.96ee5424b7af6p-23 + T * (0x1.bc128a9b8a724p-36 + T * -0x1.854ddeba4197bp-50)))) + -0x1.cd661b089a027p+9)), f[0], tmp);
      tmp = fma(-(0x1.01c2d34acaff7p+13 * (T * (0x1.40000015798eep+1 + T * (-0x1.961a6ea91e1b0p-37 + T * (0x1.840f104982ce0p-48 + T * (-0x1.5d647fca8f878p-60 + T * 0x1.e1d3b0ee8129dp-74)))) + 0x1.8e06a3bcd35a8p+14)), f[1], tmp);
      tmp = fma(-(0x1.03d2b851eb852p+8 * (T * (0x1.a42a332f575b8p+1 + T * (0x1.84c851ecf574dp-11 + T * (-0x1.0f496e2f6b32bp-22 + T * (0x1.cca17066bf423p-35 + T * -0x1.3852c0eebb013p-48)))) + -0x1.101d4b48d3ae7p+10)), f[2], tmp);
      tmp = fma(-(0x1.03d2b851eb852p+9 * (T * (0x1.48e2c7b5e1a3dp+1 + T * (-0x1.689a0073e4c12p-15 + T * (0x1.e0722e91f065fp-27 + T * (-0x1.607823b4427e2p-39 + T * 0x1.1b3c369230ddcp-52)))) + 0x1.c88650ff97247p+14)), f[3], tmp);
      tmp = fma(-(0x1.e8d949731098dp+8 * (T * (0x1.6eaf6f6ecdbe1p+1 + T * (0x1.14f4d0c23ad0ap-11 + T * (-0x1.72ead5bfa9624p-24 + T * (0x1.0c7922a4a2d04p-37 + T * -0x1.3320f7b200b9ap-52)))) + 0x1.d0db729b280f1p+11)), f[4], tmp);
      tmp = fma(-(0x1.01c2d350092cdp+12 * (T * (0x1.ab2bf6fecf7e5p+1 + T * (-0x1.9e6b00c08fd91p-16 + T * (0x1.65866c34c762ap-23 + T * (-0x1.8adee4a4b6baep-35 + T * 0x1.2099318342be3p-48)))) + -0x1.db14578e5c4ebp+9)), f[5], tmp);
      tmp = fma(-(0x1.cd7f5ff609dd0p+8 * (T * (0x1.8459ddac6e07ap+1 + T * (0x1.1d553f9364039p-10 + T * (-0x1.d5ca6d6fbef3fp-25 + T * (-0x1.aacb905b9d982p-36 + T * 0x1.e4ce6d148b330p-49)))) + -0x1.d4d1303afb7e9p+14)), f[6], tmp);
      tmp = fma(-(0x1.f7c6fae7924afp+7 * (T * (0x1.0119fbbf289f6p+2 + T * (0x1.2593e454221e1p-10 + T * (-0x1.c597157493eb4p-23 + T * (0x1.f675fa32f618cp-36 + T * -0x1.370671f4bb474p-49)))) + 0x1.bf6d462c343b7p+6)), f[7], tmp);
      tmp = fma(-(0x1.e8d94983d7907p+7 * (T * (0x1.0a8f681d1fcb7p+2 + T * (0x1.41abe4bc5704bp-9 + T * (-0x1.544474260f258p-21 + T * (0x1.981f91177d524p-34 + T * -0x1.9eeb6a97eb6fbp-48)))) + -0x1.1717269ad42c4p+14)), f[8], tmp);
    } else {
      tmp = fma(-(0x1.28ba9057d1783p+8 * (T * (0x1.a63b0c4588a05p+1 + T * (0x1.712969da04050p-11 + T * (-0x1.629f839620fc6p-20 + T * (0x1.83ae94da0fe59p-30 + T * -0x1.13441e6a0b3dfp-41)))) + -0x1.fe732fec56d5dp+9)), f[0], tmp);
      tmp = fma(-(0x1.01c2d34acaff7p+13 * (T * (0x1.4000000000000p+1 + T * (0x1.8d112bf5fb7e0p-42 + T * (-0x1.7f85eab504006p-51 + T * (0x1.538a620b2373fp-61 + T * -0x1.c09fb31fd8141p-73)))) + 0x1.8e06a3bcd35a8p+14)), f[1], tmp);
      tmp = fma(-(0x1.03d2b851eb852p+8 * (T * (0x1.e42787ae5fa45p+1 + T * (-0x1.88c9b66c8c0dfp-10 + T * (0x1.b88f92cda255fp-19 + T * (-0x1.4ca5927516966p-29 + T * 0x1.6d361ad59bca4p-41)))) + -0x1.09fc63497b741p+10)), f[2], tmp);
      tmp = fma(-(0x1.03d2b851eb852p+9 * (T * (0x1.9589c6bdbf12dp+1 + T * (-0x1.add3ae5787a18p-10 + T * (0x1.2934a57c4d958p-19 + T * (-0x1.a51e14d5c0503p-30 + T * 0x1.dbba8a635ed80p-42)))) + 0x1.c709096bb98c8p+14)), f[3], tmp);
      tmp = fma(-(0x1.e8d949731098dp+8 * (T * (0x1.080501d23d242p+2 + T * (-0x1.a6c41f6034cc8p-10 + T * (0x1.240abf1dbdb41p-19 + T * (-0x1.8e78ee8cec246p-30 + T * 0x1.d067c130d5fbcp-42)))) + 0x1.a6b138476f2a6p+11)), f[4], tmp);
      tmp = fma(-(0x1.01c2d350092cdp+12 * (T * (0x1.2c130ac9b2911p+1 + T * (0x1.058175caab342p-8 + T * (-0x1.b3b80759749d1p-18 + T * (0x1.5a4c582f87e3dp-28 + T * -0x1.9f3d0eb996c74p-40)))) + -0x1.caf7b3bfb58d1p+9)), f[5], tmp);
      tmp = fma(-(0x1.cd7f5ff609dd0p+8 * (T * (0x1.0cb686e536fbfp+2 + T * (-0x1.0aeb63b84c925p-10 + T * (0x1.23b7c52ad124bp-19 + T * (-0x1.7921668781cadp-30 + T * 0x1.8f03963eb52f4p-42)))) + -0x1.d956e8240b780p+14)), f[6], tmp);
      tmp = fma(-(0x1.f7c6fae7924afp+7 * (T * (0x1.1350a899bcaa1p+2 + T * (-0x1.373d053b75995p-9 + T * (0x1.d94d8bd675c95p-18 + T * (-0x1.a110b0905e0fcp-28 + T * 0x1.058dba115721ap-39)))) + 0x1.26cedbb59ddc2p+8)), f[7], tmp);
      tmp = fma(-(0x1.e8d94983d7907p+7 * (T * (0x1.11abd48f63e0ap+2 + T * (-0x1.1c986431acf9ep-12 + T * (0x1.7652d932e9587p-18 + T * (-0x1.72b101cd97284p-28 + T * 0x1.e584c5e48fadep-40)))) + -0x1.149a541205bc0p+14)), f[8], tmp);
    }
    f[9] = tmp / cpm;
  }
};

}  // namespace tgr
