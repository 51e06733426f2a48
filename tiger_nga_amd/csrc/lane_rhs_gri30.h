/* Generated by tiger_nga_amd/mech/lanegen.py from the compiled mechanism gri30
 * (reference combustion/grimech30F.f90).  Do not edit.  Lane-per-state right-hand side of
 * finitechem_compute_rhs (combustion/finitechem.f90:93-175). */
#pragma once
#include "lane_rhs.h"

namespace tgr {

template <>
struct LaneRhs<37> {
  // production rates cd (kmol/m3/s) from the concentrations, temperature and pressure of this lane's state
  static __device__ __forceinline__ void rates(const double (&C)[36], double T, double P, double (&cd)[36]) {
    const double C0 = C[0];
    const double C1 = C[1];
    const double C2 = C[2];
    const double C3 = C[3];
    const double C4 = C[4];
    const double C5 = C[5];
    const double C6 = C[6];
    const double C7 = C[7];
    const double C8 = C[8];
    const double C9 = C[9];
    const double C10 = C[10];
    const double C11 = C[11];
    const double C12 = C[12];
    const double C13 = C[13];
    const double C14 = C[14];
    const double C15 = C[15];
    const double C16 = C[16];
    const double C17 = C[17];
    const double C18 = C[18];
    const double C19 = C[19];
    const double C20 = C[20];
    const double C21 = C[21];
    const double C22 = C[22];
    const double C23 = C[23];
    const double C24 = C[24];
    const double C25 = C[25];
    const double C26 = C[26];
    const double C27 = C[27];
    const double C28 = C[28];
    const double C29 = C[29];
    const double C30 = C[30];
    const double C31 = C[31];
    const double C32 = C[32];
    const double C33 = C[33];
    const double C34 = C[34];
    const double C35 = C[35];
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
    ctot += C9;
    ctot += C10;
    ctot += C11;
    ctot += C12;
    ctot += C13;
    ctot += C14;
    ctot += C15;
    ctot += C16;
    ctot += C17;
    ctot += C18;
    ctot += C19;
    ctot += C20;
    ctot += C21;
    ctot += C22;
    ctot += C23;
    ctot += C24;
    ctot += C25;
    ctot += C26;
    ctot += C27;
    ctot += C28;
    ctot += C29;
    ctot += C30;
    ctot += C31;
    ctot += C32;
    ctot += C33;
    ctot += C34;
    ctot += C35;
    auto M0 = [&]() { double s_ = ctot; s_ = fma(0x1.6666680000000p+0, C5, s_); s_ = fma(0x1.8000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.4ccccc0000000p+1, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.cccccc0000000p+3, C28, s_); s_ = fma(-0x1.5c28f80000000p-3, C29, s_); return s_; };
    auto M1 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.4000000000000p+2, C28, s_); s_ = fma(-0x1.3333340000000p-2, C29, s_); return s_; };
    auto M2 = [&]() { double s_ = ctot; s_ = fma(0x1.4000000000000p+2, C2, s_); s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.4000000000000p+1, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.4000000000000p+2, C28, s_); s_ = fma(-0x1.0000000000000p-1, C29, s_); return s_; };
    auto M3 = [&]() { double s_ = ctot; s_ = fma(-0x1.0000000000000p+0, C0, s_); s_ = fma(-0x1.0000000000000p+0, C2, s_); s_ = fma(-0x1.0000000000000p-2, C9, s_); s_ = fma(0x1.0000000000000p-1, C16, s_); s_ = fma(0x1.0000000000000p-1, C27, s_); s_ = fma(-0x1.0000000000000p+0, C28, s_); s_ = fma(-0x1.0000000000000p+0, C29, s_); return s_; };
    auto M4 = [&]() { double s_ = ctot; s_ = fma(-0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(-0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(-0x1.0000000000000p+0, C28, s_); s_ = fma(-0x1.7ae1480000000p-2, C29, s_); return s_; };
    auto M5 = [&]() { double s_ = ctot; s_ = fma(-0x1.147ae00000000p-2, C5, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.5333340000000p+1, C28, s_); s_ = fma(-0x1.3d70a40000000p-1, C29, s_); return s_; };
    auto M6 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.4000000000000p+2, C28, s_); s_ = fma(-0x1.3333340000000p-2, C29, s_); return s_; };
    auto M7 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+1, C15, s_); s_ = fma(0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.4000000000000p+2, C28, s_); s_ = fma(-0x1.3333340000000p-2, C29, s_); return s_; };
    auto M8 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.4000000000000p+2, C28, s_); s_ = fma(-0x1.3333340000000p-2, C29, s_); return s_; };
    auto M9 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.4000000000000p+2, C28, s_); return s_; };
    auto M10 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.4000000000000p+2, C28, s_); return s_; };
    auto M11 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.4000000000000p+2, C28, s_); return s_; };
    auto M12 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.4000000000000p+2, C28, s_); return s_; };
    auto M13 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.4000000000000p+2, C28, s_); s_ = fma(-0x1.3333340000000p-2, C29, s_); return s_; };
    auto M14 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.4000000000000p+2, C28, s_); s_ = fma(-0x1.3333340000000p-2, C29, s_); return s_; };
    auto M15 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.4000000000000p+2, C28, s_); s_ = fma(-0x1.3333340000000p-2, C29, s_); return s_; };
    auto M16 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.4000000000000p+2, C28, s_); s_ = fma(-0x1.3333340000000p-2, C29, s_); return s_; };
    auto M17 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.4000000000000p+2, C28, s_); s_ = fma(-0x1.3333340000000p-2, C29, s_); return s_; };
    auto M18 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.4000000000000p+2, C28, s_); s_ = fma(-0x1.3333340000000p-2, C29, s_); return s_; };
    auto M19 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.4000000000000p+2, C28, s_); s_ = fma(-0x1.3333340000000p-2, C29, s_); return s_; };
    auto M20 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.4000000000000p+2, C28, s_); return s_; };
    auto M21 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.4000000000000p+2, C28, s_); s_ = fma(-0x1.3333340000000p-2, C29, s_); return s_; };
    auto M22 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.4000000000000p+2, C28, s_); s_ = fma(-0x1.3333340000000p-2, C29, s_); return s_; };
    auto M23 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.4000000000000p+2, C28, s_); return s_; };
    auto M24 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.4000000000000p+2, C28, s_); s_ = fma(-0x1.3333340000000p-2, C29, s_); return s_; };
    auto M25 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(-0x1.0000000000000p+0, C28, s_); return s_; };
    auto M26 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.4000000000000p+2, C28, s_); s_ = fma(-0x1.3333340000000p-2, C29, s_); return s_; };
    auto M27 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.4000000000000p+2, C28, s_); s_ = fma(-0x1.3333340000000p-2, C29, s_); return s_; };
    auto M28 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.4000000000000p+2, C28, s_); s_ = fma(-0x1.3333340000000p-2, C29, s_); return s_; };
    auto M29 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.4000000000000p+2, C28, s_); s_ = fma(-0x1.3333340000000p-2, C29, s_); return s_; };
    auto M30 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.4000000000000p+2, C28, s_); s_ = fma(-0x1.3333340000000p-2, C29, s_); return s_; };
    auto M31 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.0000000000000p-1, C9, s_); s_ = fma(0x1.0000000000000p+0, C15, s_); s_ = fma(0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C27, s_); s_ = fma(0x1.4000000000000p+2, C28, s_); s_ = fma(-0x1.3333340000000p-2, C29, s_); return s_; };
    double cd0 = 0.0;
    double cd1 = 0.0;
    double cd2 = 0.0;
    double cd3 = 0.0;
    double cd4 = 0.0;
    double cd5 = 0.0;
    double cd6 = 0.0;
    double cd7 = 0.0;
    double cd8 = 0.0;
    double cd9 = 0.0;
    double cd10 = 0.0;
    double cd11 = 0.0;
    double cd12 = 0.0;
    double cd13 = 0.0;
    double cd14 = 0.0;
    double cd15 = 0.0;
    double cd16 = 0.0;
    double cd17 = 0.0;
    double cd18 = 0.0;
    double cd19 = 0.0;
    double cd20 = 0.0;
    double cd21 = 0.0;
    double cd22 = 0.0;
    double cd23 = 0.0;
    double cd24 = 0.0;
    double cd25 = 0.0;
    double cd26 = 0.0;
    double cd27 = 0.0;
    double cd28 = 0.0;
    double cd29 = 0.0;
    double cd30 = 0.0;
    double cd31 = 0.0;
    double cd32 = 0.0;
    double cd33 = 0.0;
    double cd34 = 0.0;
    double cd35 = 0.0;
    {  // R3 (elementary)
    const double kf = 0x1.7d29949a6a30ap+29 * fexp2(fma(-0x1.8fa8800000000p+24, irt, 0x1.59999a0000000p+1 * lt));
    const double kb = 0x1.6c51664a92487p+28 * fexp2(fma(-0x1.174d420000000p+24, irt, 0x1.551cc20000000p+1 * lt));
    const double q = kf * C1 * C5 - kb * C4 * C3;
    cd1 -= q;
    cd3 += q;
    cd4 += q;
    cd5 -= q;
    }
    {  // R4 (elementary)
    const double kf = 0x1.2a05f20000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.ba5a6d736e7f1p+33 * fexp2(fma(-0x1.a4a3980000000p+27, irt, 0x1.4edbb60000000p-2 * lt));
    const double q = kf * C1 * C6 - kb * C2 * C4;
    cd1 -= q;
    cd2 += q;
    cd4 += q;
    cd6 -= q;
    }
    {  // R5 (elementary)
    const double kf = 0x1.2cf0000000000p+31 * fexp2(fma(-0x1.febe000000000p+23, irt, 0x1.0000000000000p+1 * lt));
    const double kb = 0x1.581e796af36cbp+27 * fexp2(fma(-0x1.20b98a0000000p+26, irt, 0x1.4934040000000p+1 * lt));
    const double q = kf * C1 * C7 - kb * C6 * C4;
    cd1 -= q;
    cd4 += q;
    cd6 += q;
    cd7 -= q;
    }
    {  // R6 (elementary)
    const double kf = 0x1.a8aedf4000000p+35 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.4a5b9d02f7e58p+41 * fexp2(fma(-0x1.608f560000000p+29, irt, -0x1.c418280000000p-5 * lt));
    const double q = kf * C1 * C8 - kb * C9 * C3;
    cd1 -= q;
    cd3 += q;
    cd8 -= q;
    cd9 += q;
    }
    {  // R7 (elementary)
    const double kf = 0x1.2a05f20000000p+36 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.a59a1fbbb39b0p+39 * fexp2(fma(-0x1.6d9ce00000000p+28, irt, -0x1.61f6440000000p-2 * lt));
    const double q = kf * C1 * C10 - kb * C11 * C3;
    cd1 -= q;
    cd3 += q;
    cd10 -= q;
    cd11 += q;
    }
    {  // R8 (elementary)
    const double kf = 0x1.bf08eb0000000p+33 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.05df9af9e2976p+37 * fexp2(fma(-0x1.77bea40000000p+29, irt, 0x1.6663c80000000p-3 * lt));
    const double q = kf * C1 * C12 - kb * C9 * C5;
    cd1 -= q;
    cd5 += q;
    cd9 += q;
    cd12 -= q;
    }
    {  // R9 (elementary)
    const double kf = 0x1.bf08eb0000000p+33 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.38a0c1550bab4p+36 * fexp2(fma(-0x1.91300c0000000p+28, irt, -0x1.a1be2c0000000p-2 * lt));
    const double q = kf * C1 * C12 - kb * C11 * C3;
    cd1 -= q;
    cd3 += q;
    cd11 += q;
    cd12 -= q;
    }
    {  // R10 (elementary)
    const double kf = 0x1.78ffd74000000p+35 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.181fdff02978fp+40 * fexp2(fma(-0x1.1380e4b000000p+28, irt, -0x1.1a61180000000p-2 * lt));
    const double q = kf * C1 * C13 - kb * C14 * C3;
    cd1 -= q;
    cd3 += q;
    cd13 -= q;
    cd14 += q;
    }
    {  // R11 (elementary)
    const double kf = 0x1.602c1d5682825p+33 * fexp2(fma(-0x1.1285580000000p+25, irt, 0x1.8000000000000p+0 * lt));
    const double kb = 0x1.2cbae9b651fccp+26 * fexp2(fma(-0x1.2262520000000p+24, irt, 0x1.f9fbe80000000p+0 * lt));
    const double q = kf * C1 * C15 - kb * C13 * C4;
    cd1 -= q;
    cd4 += q;
    cd13 += q;
    cd15 -= q;
    }
    {  // R13 (elementary)
    const double kf = 0x1.bf08eb0000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.65e78d70a7110p+34 * fexp2(fma(-0x1.56c7860000000p+28, irt, 0x1.1884400000000p-1 * lt));
    const double q = kf * C1 * C11 - kb * C9 * C4;
    cd1 -= q;
    cd4 += q;
    cd9 += q;
    cd11 -= q;
    }
    {  // R14 (elementary)
    const double kf = 0x1.bf08eb0000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.4b748c11f236dp+45 * fexp2(fma(-0x1.bf34f00000000p+28, irt, -0x1.7615a80000000p-1 * lt));
    const double q = kf * C1 * C11 - kb * C16 * C3;
    cd1 -= q;
    cd3 += q;
    cd11 -= q;
    cd16 += q;
    }
    {  // R15 (elementary)
    const double kf = 0x1.229298c000000p+35 * fexp2(fma(-0x1.c3fef00000000p+23, irt, 0.0 * lt));
    const double kb = 0x1.e8a47f391a8d3p+28 * fexp2(fma(-0x1.0c972e0000000p+26, irt, 0x1.a855da0000000p-2 * lt));
    const double q = kf * C1 * C14 - kb * C11 * C4;
    cd1 -= q;
    cd4 += q;
    cd11 += q;
    cd14 -= q;
    }
    {  // R16 (elementary)
    const double kf = 0x1.2a05f20000000p+33 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.3fdaac1a2dfdcp+33 * fexp2(fma(-0x1.206df20000000p+28, irt, 0x1.64a0c20000000p-1 * lt));
    const double q = kf * C1 * C17 - kb * C14 * C4;
    cd1 -= q;
    cd4 += q;
    cd14 += q;
    cd17 -= q;
    }
    {  // R17 (elementary)
    const double kf = 0x1.2a05f20000000p+33 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.903ff4de082abp+29 * fexp2(fma(-0x1.3ba2a80000000p+28, irt, 0x1.4661ae0000000p-1 * lt));
    const double q = kf * C1 * C18 - kb * C14 * C4;
    cd1 -= q;
    cd4 += q;
    cd14 += q;
    cd18 -= q;
    }
    {  // R18 (elementary)
    const double kf = 0x1.125b809ac6b51p+31 * fexp2(fma(-0x1.8bd0200000000p+23, irt, 0x1.4000000000000p+1 * lt));
    const double kb = 0x1.d43984f485becp+24 * fexp2(fma(-0x1.ef54200000000p+24, irt, 0x1.5685880000000p+1 * lt));
    const double q = kf * C1 * C19 - kb * C17 * C4;
    cd1 -= q;
    cd4 += q;
    cd17 += q;
    cd19 -= q;
    }
    {  // R19 (elementary)
    const double kf = 0x1.6fb20e01938bcp+29 * fexp2(fma(-0x1.3f36c00000000p+24, irt, 0x1.4000000000000p+1 * lt));
    const double kb = 0x1.f57cc83b50d01p+26 * fexp2(fma(-0x1.6aaee20000000p+23, irt, 0x1.5e15760000000p+1 * lt));
    const double q = kf * C1 * C19 - kb * C18 * C4;
    cd1 -= q;
    cd4 += q;
    cd18 += q;
    cd19 -= q;
    }
    {  // R20 (elementary)
    const double kf = 0x1.74876e8000000p+35 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.81b31c759932bp+33 * fexp2(fma(-0x1.3689680000000p+28, irt, 0x1.033c600000000p+0 * lt));
    const double q = kf * C1 * C20 - kb * C9 * C8;
    cd1 -= q;
    cd8 += q;
    cd9 += q;
    cd20 -= q;
    }
    {  // R21 (elementary)
    const double kf = 0x1.a5e0000000000p+31 * fexp2(fma(-0x1.e53ac00000000p+22, irt, 0x1.0000000000000p+1 * lt));
    const double kb = 0x1.a1ff8b270f30dp+31 * fexp2(fma(-0x1.566c7e0000000p+26, irt, 0x1.d167240000000p+0 * lt));
    const double q = kf * C1 * C21 - kb * C22 * C3;
    cd1 -= q;
    cd3 += q;
    cd21 -= q;
    cd22 += q;
    }
    {  // R22 (elementary)
    const double kf = 0x1.9532b82aeba9ap+42 * fexp2(fma(-0x1.ce10160000000p+26, irt, -0x1.68f5c20000000p+0 * lt));
    const double kb = 0x1.5e6ecf2456a80p+35 * fexp2(fma(0x1.35d0f00000000p+23, irt, -0x1.b271bc0000000p-1 * lt));
    const double q = kf * C1 * C21 - kb * C20 * C4;
    cd1 -= q;
    cd4 += q;
    cd20 += q;
    cd21 -= q;
    }
    {  // R23 (elementary)
    const double kf = 0x1.b1c0000000000p+30 * fexp2(fma(-0x1.e53ac00000000p+22, irt, 0x1.0000000000000p+1 * lt));
    const double kb = 0x1.0ac46a80b3038p+24 * fexp2(fma(-0x1.7b4c1c0000000p+27, irt, 0x1.a88a480000000p+1 * lt));
    const double q = kf * C1 * C21 - kb * C10 * C9;
    cd1 -= q;
    cd9 += q;
    cd10 += q;
    cd21 -= q;
    }
    {  // R24 (elementary)
    const double kf = 0x1.bf08eb0000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.5d3650437691bp+41 * fexp2(fma(-0x1.698393d000000p+28, irt, -0x1.33a0a60000000p-1 * lt));
    const double q = kf * C1 * C23 - kb * C24 * C3;
    cd1 -= q;
    cd3 += q;
    cd23 -= q;
    cd24 += q;
    }
    {  // R25 (elementary)
    const double kf = 0x1.0e877df03698bp+30 * fexp2(fma(-0x1.c138000000000p+19, irt, 0x1.d47ae20000000p+0 * lt));
    const double kb = 0x1.8096187af61c2p+21 * fexp2(fma(-0x1.9d6be40000000p+26, irt, 0x1.5ab4640000000p+1 * lt));
    const double q = kf * C1 * C25 - kb * C11 * C13;
    cd1 -= q;
    cd11 += q;
    cd13 += q;
    cd25 -= q;
    }
    {  // R26 (elementary)
    const double kf = 0x1.4dc9380000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.3fa056f367921p+32 * fexp2(fma(-0x1.36a2640000000p+28, irt, 0x1.cd2bf60000000p-1 * lt));
    const double q = kf * C1 * C26 - kb * C14 * C13;
    cd1 -= q;
    cd13 += q;
    cd14 += q;
    cd26 -= q;
    }
    {  // R27 (elementary)
    const double kf = 0x1.a9eaabe2b355ep+33 * fexp2(fma(-0x1.6b44180000000p+24, irt, 0x1.eb851e0000000p+0 * lt));
    const double kb = 0x1.40de405676d9fp+25 * fexp2(fma(-0x1.a11cd40000000p+24, irt, 0x1.38d8ec0000000p+1 * lt));
    const double q = kf * C1 * C27 - kb * C26 * C4;
    cd1 -= q;
    cd4 += q;
    cd26 += q;
    cd27 -= q;
    }
    {  // R28 (elementary)
    const double kf = 0x1.74876e8000000p+36 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.0e14604f5a06bp+23 * fexp2(fma(-0x1.96edce0000000p+28, irt, 0x1.62c27a0000000p+0 * lt));
    const double q = kf * C1 * C22 - kb * C9 * C9 * C3;
    cd1 -= q;
    cd3 += q;
    cd9 = fma(0x1.0000000000000p+1, q, cd9);
    cd22 -= q;
    }
    {  // R29 (elementary)
    const double kf = 0x1.2a05f20000000p+33 * fexp2(fma(-0x1.febe000000000p+24, irt, 0.0 * lt));
    const double kb = 0x1.21db7dca1f62bp+27 * fexp2(fma(-0x1.bdfc340000000p+23, irt, 0x1.1fcc7e0000000p-1 * lt));
    const double q = kf * C1 * C24 - kb * C22 * C4;
    cd1 -= q;
    cd4 += q;
    cd22 += q;
    cd24 -= q;
    }
    {  // R30 (elementary)
    const double kf = 0x1.a13b860000000p+30 * fexp2(fma(-0x1.58ba000000000p+22, irt, 0.0 * lt));
    const double kb = 0x1.d288008e31fa5p+28 * fexp2(fma(-0x1.87be860000000p+27, irt, 0x1.908c600000000p-1 * lt));
    const double q = kf * C1 * C24 - kb * C16 * C10;
    cd1 -= q;
    cd10 += q;
    cd16 += q;
    cd24 -= q;
    }
    {  // R31 (elementary)
    const double kf = 0x1.2a05f20000000p+31 * fexp2(fma(-0x1.7d75cf0000000p+27, irt, 0.0 * lt));
    const double kb = 0x1.0b25be078e7aap+37 * fexp2(fma(-0x1.c3ce520000000p+27, irt, -0x1.aef5ec0000000p-1 * lt));
    const double q = kf * C2 * C9 - kb * C16 * C1;
    cd1 += q;
    cd2 -= q;
    cd9 -= q;
    cd16 += q;
    }
    {  // R32 (elementary)
    const double kf = 0x1.74876e8000000p+36 * fexp2(fma(-0x1.3f36c00000000p+27, irt, 0.0 * lt));
    const double kb = 0x1.a61046d5b85f3p+30 * fexp2(fma(-0x1.27b4460000000p+21, irt, 0x1.65e8ac0000000p-4 * lt));
    const double q = kf * C2 * C14 - kb * C11 * C6;
    cd2 -= q;
    cd6 += q;
    cd11 += q;
    cd14 -= q;
    }
    {  // R34 (elementary)
    const double kf = 0x1.0ee7f155e7f91p+33 * fexp2(fma(0.0, irt, -0x1.3d70a40000000p+0 * lt));
    const double kb = 0x1.61f66018d96ebp+43 * fexp2(fma(-0x1.865f740000000p+27, irt, -0x1.4078960000000p+0 * lt));
    const double q = kf * C3 * C2 * C2 - kb * C2 * C6;
    cd2 -= q;
    cd3 -= q;
    cd6 += q;
    }
    {  // R35 (elementary)
    const double kf = 0x1.6e252d0f6ab94p+36 * fexp2(fma(0.0, irt, -0x1.851eb80000000p-1 * lt));
    const double kb = 0x1.de675107cb552p+46 * fexp2(fma(-0x1.865f740000000p+27, irt, -0x1.8b2e7c0000000p-1 * lt));
    const double q = kf * C3 * C2 * C28 - kb * C28 * C6;
    cd2 -= q;
    cd3 -= q;
    cd6 += q;
    }
    {  // R36 (elementary)
    const double kf = 0x1.52a1edab61f76p+33 * fexp2(fma(0.0, irt, -0x1.3d70a40000000p+0 * lt));
    const double kb = 0x1.ba73f81f1c79ap+43 * fexp2(fma(-0x1.865f740000000p+27, irt, -0x1.4078960000000p+0 * lt));
    const double q = kf * C3 * C2 * C0 - kb * C0 * C6;
    cd2 -= q;
    cd3 -= q;
    cd6 += q;
    }
    {  // R37 (elementary)
    const double kf = 0x1.1bc464fefab51p+32 * fexp2(fma(0.0, irt, -0x1.99999a0000000p-1 * lt));
    const double kb = 0x1.72c4d9f7e4336p+42 * fexp2(fma(-0x1.865f740000000p+27, irt, -0x1.9fa95c0000000p-1 * lt));
    const double q = kf * C3 * C2 * C29 - kb * C29 * C6;
    cd2 -= q;
    cd3 -= q;
    cd6 += q;
    }
    {  // R38 (elementary)
    const double kf = 0x1.775742e43279dp+38 * fexp2(fma(-0x1.0ffce80000000p+26, irt, -0x1.578d500000000p-1 * lt));
    const double kb = 0x1.6b4d95f421057p+33 * fexp2(fma(0x1.41eff60000000p+20, irt, -0x1.dfa54c0000000p-3 * lt));
    const double q = kf * C3 * C2 - kb * C4 * C1;
    cd1 += q;
    cd2 -= q;
    cd3 -= q;
    cd4 += q;
    }
    {  // R40 (elementary)
    const double kf = 0x1.fc2efa228911cp+30 * fexp2(fma(0.0, irt, -0x1.3333340000000p-1 * lt));
    const double kb = 0x1.01c987be36767p+42 * fexp2(fma(-0x1.9d073a0000000p+28, irt, -0x1.ff84ca0000000p-3 * lt));
    const double q = kf * C3 * C3 * C5 - kb * C5 * C5;
    cd3 = fma(-0x1.0000000000000p+1, q, cd3);
    cd5 += q;
    }
    {  // R41 (elementary)
    const double kf = 0x1.6f197f6b68b70p+34 * fexp2(fma(0.0, irt, -0x1.4000000000000p+0 * lt));
    const double kb = 0x1.7470445440994p+45 * fexp2(fma(-0x1.9d073a0000000p+28, irt, -0x1.ccae000000000p-1 * lt));
    const double q = kf * C3 * C3 * C28 - kb * C28 * C5;
    cd3 = fma(-0x1.0000000000000p+1, q, cd3);
    cd5 += q;
    }
    {  // R42 (elementary)
    const double kf = 0x1.f438daa060000p+30 * fexp2(fma(0.0, irt, -0x1.0000000000000p+1 * lt));
    const double kb = 0x1.fb7b337fe2159p+41 * fexp2(fma(-0x1.9d073a0000000p+28, irt, -0x1.a657540000000p+0 * lt));
    const double q = kf * C3 * C3 * C16 - kb * C16 * C5;
    cd3 = fma(-0x1.0000000000000p+1, q, cd3);
    cd5 += q;
    }
    {  // R44 (elementary)
    const double kf = 0x1.d942c90000000p+31 * fexp2(fma(-0x1.56a6c00000000p+21, irt, 0.0 * lt));
    const double kb = 0x1.005fb2a02b18ep+30 * fexp2(fma(-0x1.aa34ca0000000p+27, irt, 0x1.6358b00000000p-1 * lt));
    const double q = kf * C3 * C6 - kb * C28 * C1;
    cd1 += q;
    cd3 -= q;
    cd6 -= q;
    cd28 += q;
    }
    {  // R45 (elementary)
    const double kf = 0x1.4dc9380000000p+35 * fexp2(fma(-0x1.10c4200000000p+22, irt, 0.0 * lt));
    const double kb = 0x1.032d18585d3a8p+36 * fexp2(fma(-0x1.bc35200000000p+27, irt, 0x1.72c3440000000p-2 * lt));
    const double q = kf * C3 * C6 - kb * C5 * C2;
    cd2 += q;
    cd3 -= q;
    cd5 += q;
    cd6 -= q;
    }
    {  // R46 (elementary)
    const double kf = 0x1.38eca48000000p+36 * fexp2(fma(-0x1.4457400000000p+21, irt, 0.0 * lt));
    const double kb = 0x1.c19315ee1c53dp+30 * fexp2(fma(-0x1.1f32a00000000p+27, irt, 0x1.8711d80000000p-1 * lt));
    const double q = kf * C3 * C6 - kb * C4 * C4;
    cd3 -= q;
    cd4 = fma(0x1.0000000000000p+1, q, cd4);
    cd6 -= q;
    }
    {  // R47 (elementary)
    const double kf = 0x1.7a20000000000p+31 * fexp2(fma(-0x1.4bfc480000000p+24, irt, 0x1.0000000000000p+1 * lt));
    const double kb = 0x1.c45fd1fbe8546p+28 * fexp2(fma(-0x1.51f7ac0000000p+26, irt, 0x1.4db0de0000000p+1 * lt));
    const double q = kf * C3 * C7 - kb * C5 * C6;
    cd3 -= q;
    cd5 += q;
    cd6 += q;
    cd7 -= q;
    }
    {  // R48 (elementary)
    const double kf = 0x1.2a05f20000000p+33 * fexp2(fma(-0x1.cba7e00000000p+23, irt, 0.0 * lt));
    const double kb = 0x1.7134f3892c9c4p+27 * fexp2(fma(-0x1.1902ca0000000p+28, irt, 0x1.4413fe0000000p+0 * lt));
    const double q = kf * C3 * C7 - kb * C28 * C4;
    cd3 -= q;
    cd4 += q;
    cd7 -= q;
    cd28 += q;
    }
    {  // R49 (elementary)
    const double kf = 0x1.3356219000000p+37 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.52445c8de1bdcp+38 * fexp2(fma(-0x1.73898a0000000p+26, irt, 0x1.e017980000000p-3 * lt));
    const double q = kf * C3 * C8 - kb * C5 * C30;
    cd3 -= q;
    cd5 += q;
    cd8 -= q;
    cd30 += q;
    }
    {  // R51 (elementary)
    const double kf = 0x1.bf08eb0000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.50a4e34f56fe2p+32 * fexp2(fma(-0x1.72f4c40000000p+25, irt, 0x1.d769aa0000000p-3 * lt));
    const double q = kf * C3 * C12 - kb * C5 * C8;
    cd3 -= q;
    cd5 += q;
    cd8 += q;
    cd12 -= q;
    }
    {  // R53 (elementary)
    const double kf = 0x1.e1bd1111ffb19p+33 * fexp2(fma(-0x1.5a07fc0000000p+25, irt, 0x1.9eb8520000000p+0 * lt));
    const double kb = 0x1.ae6407f263c42p+27 * fexp2(fma(-0x1.14e16c0000000p+25, irt, 0x1.10d6f60000000p+1 * lt));
    const double q = kf * C3 * C15 - kb * C5 * C13;
    cd3 -= q;
    cd5 += q;
    cd13 += q;
    cd15 -= q;
    }
    {  // R55 (elementary)
    const double kf = 0x1.116fb1e000000p+36 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.ca16c8575c033p+36 * fexp2(fma(-0x1.5e4d3a0000000p+28, irt, 0x1.2a78080000000p-1 * lt));
    const double q = kf * C3 * C11 - kb * C9 * C5;
    cd3 -= q;
    cd5 += q;
    cd9 += q;
    cd11 -= q;
    }
    {  // R58 (elementary)
    const double kf = 0x1.e09f93403f5d2p+32 * fexp2(fma(-0x1.5e20d00000000p+23, irt, 0x1.e666660000000p+0 * lt));
    const double kb = 0x1.a6ce6c32cbb98p+27 * fexp2(fma(-0x1.1df23a0000000p+26, irt, 0x1.2cbac80000000p+1 * lt));
    const double q = kf * C3 * C14 - kb * C5 * C11;
    cd3 -= q;
    cd5 += q;
    cd11 += q;
    cd14 -= q;
    }
    {  // R60 (elementary)
    const double kf = 0x1.2a05f20000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.4ea638f5d0132p+35 * fexp2(fma(-0x1.27f3a60000000p+28, irt, 0x1.76948a0000000p-1 * lt));
    const double q = kf * C3 * C17 - kb * C14 * C5;
    cd3 -= q;
    cd5 += q;
    cd14 += q;
    cd17 -= q;
    }
    {  // R61 (elementary)
    const double kf = 0x1.1ba28006d2a53p+33 * fexp2(fma(0x1.220a000000000p+20, irt, 0x1.4ccccc0000000p-1 * lt));
    const double kb = 0x1.99af9b134123bp+28 * fexp2(fma(-0x1.79606a0000000p+23, irt, 0x1.9f4f0e0000000p+0 * lt));
    const double q = kf * C3 * C17 - kb * C13 * C4;
    cd3 -= q;
    cd4 += q;
    cd13 += q;
    cd17 -= q;
    }
    {  // R62 (elementary)
    const double kf = 0x1.16c75b7ab6bb9p+34 * fexp2(fma(-0x1.3786000000000p+21, irt, -0x1.70a3d80000000p-4 * lt));
    const double kb = 0x1.0f48debe4b33ap+29 * fexp2(fma(-0x1.81e7780000000p+23, irt, 0x1.5beea20000000p+0 * lt));
    const double q = kf * C3 * C17 - kb * C28 * C12;
    cd3 -= q;
    cd12 += q;
    cd17 -= q;
    cd28 += q;
    }
    {  // R64 (elementary)
    const double kf = 0x1.01ed86b4395c7p+30 * fexp2(fma(-0x1.eb55400000000p+22, irt, 0x1.a147ae0000000p+0 * lt));
    const double kb = 0x1.42c4b041c9ffdp+26 * fexp2(fma(-0x1.1710580000000p+25, irt, 0x1.9228780000000p+0 * lt));
    const double q = kf * C3 * C18 - kb * C17 * C3;
    cd17 += q;
    cd18 -= q;
    }
    {  // R65 (elementary)
    const double kf = 0x1.2a05f20000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.a2c382ccc1503p+31 * fexp2(fma(-0x1.43285c0000000p+28, irt, 0x1.5855760000000p-1 * lt));
    const double q = kf * C3 * C18 - kb * C14 * C5;
    cd3 -= q;
    cd5 += q;
    cd14 += q;
    cd18 -= q;
    }
    {  // R66 (elementary)
    const double kf = 0x1.f9c31e5e3d12fp+34 * fexp2(fma(0x1.c138000000000p+18, irt, 0x1.0000000000000p-1 * lt));
    const double kb = 0x1.c916aa662cd52p+26 * fexp2(fma(-0x1.3d8baa0000000p+25, irt, 0x1.69c9700000000p+0 * lt));
    const double q = kf * C3 * C18 - kb * C13 * C4;
    cd3 -= q;
    cd4 += q;
    cd13 += q;
    cd18 -= q;
    }
    {  // R67 (elementary)
    const double kf = 0x1.d0e6558df896ap+35 * fexp2(fma(-0x1.1141200000000p+22, irt, -0x1.d70a3e0000000p-3 * lt));
    const double kb = 0x1.1b0c59e1dfadap+27 * fexp2(fma(-0x1.48cf500000000p+25, irt, 0x1.28f7ba0000000p+0 * lt));
    const double q = kf * C3 * C18 - kb * C28 * C12;
    cd3 -= q;
    cd12 += q;
    cd18 -= q;
    cd28 += q;
    }
    {  // R68 (elementary)
    const double kf = 0x1.efac694ea8ddbp+32 * fexp2(fma(-0x1.36e9c00000000p+24, irt, 0x1.0ccccc0000000p+1 * lt));
    const double kb = 0x1.ba8c28aa8d92cp+27 * fexp2(fma(-0x1.6c58860000000p+25, irt, 0x1.27cf800000000p+1 * lt));
    const double q = kf * C3 * C19 - kb * C5 * C17;
    cd3 -= q;
    cd5 += q;
    cd17 += q;
    cd19 -= q;
    }
    {  // R69 (elementary)
    const double kf = 0x1.e9d78f38a6e11p+30 * fexp2(fma(-0x1.36e9c00000000p+24, irt, 0x1.0ccccc0000000p+1 * lt));
    const double kb = 0x1.5d7c06c1f36cdp+29 * fexp2(fma(-0x1.2565ae0000000p+24, irt, 0x1.2f5f1c0000000p+1 * lt));
    const double q = kf * C3 * C19 - kb * C5 * C18;
    cd3 -= q;
    cd5 += q;
    cd18 += q;
    cd19 -= q;
    }
    {  // R73 (elementary)
    const double kf = 0x1.bf08eb0000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.66a4b3919dba1p+36 * fexp2(fma(-0x1.110714a000000p+28, irt, 0x1.6d43d00000000p-3 * lt));
    const double q = kf * C3 * C23 - kb * C21 * C5;
    cd3 -= q;
    cd5 += q;
    cd21 += q;
    cd23 -= q;
    }
    {  // R75 (elementary)
    const double kf = 0x1.1a6f6d08e9166p+33 * fexp2(fma(-0x1.86b7700000000p+25, irt, 0x1.43d70a0000000p+1 * lt));
    const double kb = 0x1.3af8514c94d7dp+26 * fexp2(fma(-0x1.0f5da60000000p+24, irt, 0x1.8208080000000p+1 * lt));
    const double q = kf * C3 * C25 - kb * C5 * C23;
    cd3 -= q;
    cd5 += q;
    cd23 += q;
    cd25 -= q;
    }
    {  // R77 (elementary)
    const double kf = 0x1.dcd6500000000p+30 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.1a8eb065a5bf6p+32 * fexp2(fma(-0x1.0cb3900000000p+28, irt, 0x1.e2dd7a0000000p-2 * lt));
    const double q = kf * C3 * C26 - kb * C25 * C5;
    cd3 -= q;
    cd5 += q;
    cd25 += q;
    cd26 -= q;
    }
    {  // R78 (elementary)
    const double kf = 0x1.e175ee0b49494p+33 * fexp2(fma(-0x1.e0be500000000p+24, irt, 0x1.e666660000000p+0 * lt));
    const double kb = 0x1.7b7bc86e19a55p+26 * fexp2(fma(-0x1.4779260000000p+25, irt, 0x1.3ac66a0000000p+1 * lt));
    const double q = kf * C3 * C27 - kb * C5 * C26;
    cd3 -= q;
    cd5 += q;
    cd26 += q;
    cd27 -= q;
    }
    {  // R79 (elementary)
    const double kf = 0x1.74876e8000000p+36 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.d3bfa6411ce3ap+30 * fexp2(fma(-0x1.11df060000000p+26, irt, 0x1.8f9f020000000p+0 * lt));
    const double q = kf * C3 * C22 - kb * C9 * C12;
    cd3 -= q;
    cd9 += q;
    cd12 += q;
    cd22 -= q;
    }
    {  // R80 (elementary)
    const double kf = 0x1.74876e8000000p+35 * fexp2(fma(-0x1.febe000000000p+24, irt, 0.0 * lt));
    const double kb = 0x1.7b14c1e3a8cb8p+30 * fexp2(fma(-0x1.5759560000000p+24, irt, 0x1.31c0440000000p-1 * lt));
    const double q = kf * C3 * C24 - kb * C5 * C22;
    cd3 -= q;
    cd5 += q;
    cd22 += q;
    cd24 -= q;
    }
    {  // R81 (elementary)
    const double kf = 0x1.50c4288000000p+33 * fexp2(fma(-0x1.b5b6b00000000p+23, irt, 0.0 * lt));
    const double kb = 0x1.cc5430c80139bp+25 * fexp2(fma(-0x1.11a5980000000p+27, irt, 0x1.9398200000000p+0 * lt));
    const double q = kf * C3 * C24 - kb * C9 * C13;
    cd3 -= q;
    cd9 += q;
    cd13 += q;
    cd24 -= q;
    }
    {  // R82 (elementary)
    const double kf = 0x1.2a05f20000000p+33 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.1ff34a958a9fcp+32 * fexp2(fma(-0x1.dfd95c0000000p+26, irt, 0x1.a4dec20000000p-2 * lt));
    const double q = kf * C3 * C31 - kb * C24 * C3;
    cd24 += q;
    cd31 -= q;
    }
    {  // R84 (elementary)
    const double kf = 0x1.3d8351cc599e2p+31 * fexp2(fma(-0x1.b5f5300000000p+23, irt, 0x1.828f5c0000000p+0 * lt));
    const double kb = 0x1.c9b3288e27e2ap+33 * fexp2(fma(-0x1.2e19ae0000000p+26, irt, 0x1.67b8900000000p+0 * lt));
    const double q = kf * C4 * C5 - kb * C28 * C3;
    cd3 += q;
    cd4 -= q;
    cd5 -= q;
    cd28 += q;
    }
    {  // R86 (elementary)
    const double kf = 0x1.b0e38f8935c28p+26 * fexp2(fma(0x1.0d68c00000000p+23, irt, 0x1.3333340000000p+1 * lt));
    const double kb = 0x1.46744c17a3531p+30 * fexp2(fma(-0x1.e7897e0000000p+25, irt, 0x1.2a44fa0000000p+1 * lt));
    const double q = kf * C4 * C4 - kb * C28 * C1;
    cd1 += q;
    cd4 = fma(-0x1.0000000000000p+1, q, cd4);
    cd28 += q;
    }
    {  // R87 (elementary)
    const double kf = 0x1.b022388000000p+33 * fexp2(fma(0x1.febe000000000p+20, irt, 0.0 * lt));
    const double kb = 0x1.e3b3bb98bbec4p+36 * fexp2(fma(-0x1.15af840000000p+28, irt, 0x1.0769660000000p-2 * lt));
    const double q = kf * C4 * C6 - kb * C28 * C2;
    cd2 += q;
    cd4 -= q;
    cd6 -= q;
    cd28 += q;
    }
    {  // R88 (elementary)
    const double kf = 0x1.dcd6500000000p+30 * fexp2(fma(-0x1.b447800000000p+20, irt, 0.0 * lt));
    const double kb = 0x1.9b2eeda8c4d4bp+30 * fexp2(fma(-0x1.fd24c00000000p+26, irt, 0x1.0116880000000p-1 * lt));
    const double q = kf * C4 * C7 - kb * C28 * C6;
    cd4 -= q;
    cd6 += q;
    cd7 -= q;
    cd28 += q;
    }
    {  // R89 (elementary)
    const double kf = 0x1.8289060790000p+50 * fexp2(fma(-0x1.d566fe0000000p+26, irt, 0.0 * lt));
    const double kb = 0x1.4d50918cfb087p+50 * fexp2(fma(-0x1.e5dd500000000p+27, irt, 0x1.0116880000000p-1 * lt));
    const double q = kf * C4 * C7 - kb * C28 * C6;
    cd4 -= q;
    cd6 += q;
    cd7 -= q;
    cd28 += q;
    }
    {  // R90 (elementary)
    const double kf = 0x1.74876e8000000p+35 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.1377a2e1861cep+41 * fexp2(fma(-0x1.35e1000000000p+29, irt, -0x1.04a7720000000p-2 * lt));
    const double q = kf * C4 * C30 - kb * C9 * C3;
    cd3 += q;
    cd4 -= q;
    cd9 += q;
    cd30 -= q;
    }
    {  // R91 (elementary)
    const double kf = 0x1.bf08eb0000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.b258a5514b2d7p+40 * fexp2(fma(-0x1.6a57280000000p+28, irt, -0x1.34c5b80000000p-1 * lt));
    const double q = kf * C4 * C8 - kb * C11 * C3;
    cd3 += q;
    cd4 -= q;
    cd8 -= q;
    cd11 += q;
    }
    {  // R92 (elementary)
    const double kf = 0x1.2a05f20000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.f569dd74efe32p+43 * fexp2(fma(-0x1.38970c0000000p+28, irt, -0x1.8526100000000p-1 * lt));
    const double q = kf * C4 * C10 - kb * C14 * C3;
    cd3 += q;
    cd4 -= q;
    cd10 -= q;
    cd14 += q;
    }
    {  // R93 (elementary)
    const double kf = 0x1.6120000000000p+31 * fexp2(fma(-0x1.7f0e800000000p+23, irt, 0x1.0000000000000p+1 * lt));
    const double kb = 0x1.83b877a268e99p+32 * fexp2(fma(-0x1.526a880000000p+26, irt, 0x1.1804420000000p+1 * lt));
    const double q = kf * C4 * C10 - kb * C28 * C8;
    cd4 -= q;
    cd8 += q;
    cd10 -= q;
    cd28 += q;
    }
    {  // R94 (elementary)
    const double kf = 0x1.bf08eb0000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.73cecfa738c6bp+43 * fexp2(fma(-0x1.5c2a380000000p+28, irt, -0x1.a50a240000000p-1 * lt));
    const double q = kf * C4 * C12 - kb * C14 * C3;
    cd3 += q;
    cd4 -= q;
    cd12 -= q;
    cd14 += q;
    }
    {  // R96 (elementary)
    const double kf = 0x1.20a47438ebc8ep+30 * fexp2(fma(-0x1.5a06080000000p+24, irt, 0x1.99999a0000000p+0 * lt));
    const double kb = 0x1.8084ae7c2c169p+28 * fexp2(fma(-0x1.af357e0000000p+25, irt, 0x1.01dbca0000000p+1 * lt));
    const double q = kf * C4 * C13 - kb * C28 * C10;
    cd4 -= q;
    cd10 += q;
    cd13 -= q;
    cd28 += q;
    }
    {  // R97 (elementary)
    const double kf = 0x1.18ed6c6cf0030p+37 * fexp2(fma(-0x1.69e0a00000000p+22, irt, -0x1.570a3e0000000p+0 * lt));
    const double kb = 0x1.7a86a13bd44b8p+36 * fexp2(fma(-0x1.2d52740000000p+21, irt, -0x1.b9f42c0000000p-1 * lt));
    const double q = kf * C4 * C13 - kb * C28 * C12;
    cd4 -= q;
    cd12 += q;
    cd13 -= q;
    cd28 += q;
    }
    {  // R98 (elementary)
    const double kf = 0x1.01b767c51baa3p+31 * fexp2(fma(-0x1.8e60600000000p+23, irt, 0x1.99999a0000000p+0 * lt));
    const double kb = 0x1.4be782895874ep+27 * fexp2(fma(-0x1.0693cc0000000p+26, irt, 0x1.00dc340000000p+1 * lt));
    const double q = kf * C4 * C15 - kb * C28 * C13;
    cd4 -= q;
    cd13 += q;
    cd15 -= q;
    cd28 += q;
    }
    {  // R99 (elementary)
    const double kf = 0x1.8185f8f01b45cp+26 * fexp2(fma(-0x1.1e22000000000p+18, irt, 0x1.3a5e360000000p+0 * lt));
    const double kb = 0x1.65085b66a8d8dp+37 * fexp2(fma(-0x1.a2d3ce0000000p+26, irt, -0x1.9dd8220000000p-5 * lt));
    const double q = kf * C4 * C9 - kb * C16 * C3;
    cd3 += q;
    cd4 -= q;
    cd9 -= q;
    cd16 += q;
    }
    {  // R100 (elementary)
    const double kf = 0x1.74876e8000000p+35 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.c1d6afee6d028p+38 * fexp2(fma(-0x1.9c23fc0000000p+28, irt, 0x1.e996320000000p-2 * lt));
    const double q = kf * C4 * C11 - kb * C9 * C28;
    cd4 -= q;
    cd9 += q;
    cd11 -= q;
    cd28 += q;
    }
    {  // R101 (elementary)
    const double kf = 0x1.41bee09672314p+32 * fexp2(fma(0x1.c88b000000000p+20, irt, 0x1.2e147a0000000p+0 * lt));
    const double kb = 0x1.98088b5efbc99p+29 * fexp2(fma(-0x1.e266fc0000000p+26, irt, 0x1.864d800000000p+0 * lt));
    const double q = kf * C4 * C14 - kb * C28 * C11;
    cd4 -= q;
    cd11 += q;
    cd14 -= q;
    cd28 += q;
    }
    {  // R102 (elementary)
    const double kf = 0x1.2a05f20000000p+32 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.e26a11bbd565bp+35 * fexp2(fma(-0x1.65ca680000000p+28, irt, 0x1.40e77a0000000p-1 * lt));
    const double q = kf * C4 * C17 - kb * C14 * C28;
    cd4 -= q;
    cd14 += q;
    cd17 -= q;
    cd28 += q;
    }
    {  // R103 (elementary)
    const double kf = 0x1.2a05f20000000p+32 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.2dd62ba0de80ep+32 * fexp2(fma(-0x1.80ff1e0000000p+28, irt, 0x1.22a8860000000p-1 * lt));
    const double q = kf * C4 * C18 - kb * C14 * C28;
    cd4 -= q;
    cd14 += q;
    cd18 -= q;
    cd28 += q;
    }
    {  // R104 (elementary)
    const double kf = 0x1.6800000000000p+28 * fexp2(fma(0x1.ad13c00000000p+21, irt, 0x1.0000000000000p+1 * lt));
    const double kb = 0x1.cf53456e5ef51p+25 * fexp2(fma(-0x1.52643e0000000p+26, irt, 0x1.0d974e0000000p+1 * lt));
    const double q = kf * C4 * C19 - kb * C28 * C17;
    cd4 -= q;
    cd17 += q;
    cd19 -= q;
    cd28 += q;
    }
    {  // R105 (elementary)
    const double kf = 0x1.89c0000000000p+30 * fexp2(fma(-0x1.7f0e800000000p+22, irt, 0x1.0000000000000p+1 * lt));
    const double kb = 0x1.94fc22aa496ddp+31 * fexp2(fma(-0x1.0aeaec0000000p+26, irt, 0x1.15273e0000000p+1 * lt));
    const double q = kf * C4 * C19 - kb * C28 * C18;
    cd4 -= q;
    cd18 += q;
    cd19 -= q;
    cd28 += q;
    }
    {  // R106 (elementary)
    const double kf = 0x1.2a05f20000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.55700303ab9a6p+41 * fexp2(fma(-0x1.9671840000000p+27, irt, -0x1.7cab1e0000000p-1 * lt));
    const double q = kf * C4 * C20 - kb * C22 * C3;
    cd3 += q;
    cd4 -= q;
    cd20 -= q;
    cd22 += q;
    }
    {  // R107 (elementary)
    const double kf = 0x1.4b0876427145fp+18 * fexp2(fma(0x1.febe000000000p+21, irt, 0x1.2000000000000p+2 * lt));
    const double kb = 0x1.513f012c724dcp+24 * fexp2(fma(-0x1.7012dc0000000p+26, irt, 0x1.e0c0ae0000000p+1 * lt));
    const double q = kf * C4 * C21 - kb * C24 * C3;
    cd3 += q;
    cd4 -= q;
    cd21 -= q;
    cd24 += q;
    }
    {  // R108 (elementary)
    const double kf = 0x1.996005a2a44c1p+29 * fexp2(fma(-0x1.aef0500000000p+25, irt, 0x1.2666660000000p+1 * lt));
    const double kb = 0x1.afa30d39146c8p+36 * fexp2(fma(-0x1.de9e640000000p+24, irt, 0x1.2516340000000p+0 * lt));
    const double q = kf * C4 * C21 - kb * C31 * C3;
    cd3 += q;
    cd4 -= q;
    cd21 -= q;
    cd31 += q;
    }
    {  // R109 (elementary)
    const double kf = 0x1.0748000000000p+33 * fexp2(fma(-0x1.bee6400000000p+25, irt, 0x1.0000000000000p+1 * lt));
    const double kb = 0x1.5769cc5804311p+29 * fexp2(fma(-0x1.ac37220000000p+14, irt, 0x1.3ef0060000000p+1 * lt));
    const double q = kf * C4 * C21 - kb * C28 * C20;
    cd4 -= q;
    cd20 += q;
    cd21 -= q;
    cd28 += q;
    }
    {  // R110 (elementary)
    const double kf = 0x1.034f03b80a36dp+15 * fexp2(fma(0x1.febe000000000p+22, irt, 0x1.0000000000000p+2 * lt));
    const double kb = 0x1.691a7a26114b4p+13 * fexp2(fma(-0x1.a658a20000000p+27, irt, 0x1.35465e0000000p+2 * lt));
    const double q = kf * C4 * C21 - kb * C9 * C13;
    cd4 -= q;
    cd9 += q;
    cd13 += q;
    cd21 -= q;
    }
    {  // R111 (elementary)
    const double kf = 0x1.2a05f20000000p+32 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.58ab73966481bp+36 * fexp2(fma(-0x1.4eddd60000000p+28, irt, 0x1.2d1fa40000000p-4 * lt));
    const double q = kf * C4 * C23 - kb * C21 * C28;
    cd4 -= q;
    cd21 += q;
    cd23 -= q;
    cd28 += q;
    }
    {  // R112 (elementary)
    const double kf = 0x1.c200000000000p+29 * fexp2(fma(-0x1.3f36c00000000p+23, irt, 0x1.0000000000000p+1 * lt));
    const double kb = 0x1.69b3f5f94c252p+25 * fexp2(fma(-0x1.3f7b240000000p+25, irt, 0x1.30c5980000000p+1 * lt));
    const double q = kf * C4 * C25 - kb * C28 * C23;
    cd4 -= q;
    cd23 += q;
    cd25 -= q;
    cd28 += q;
    }
    {  // R113 (elementary)
    const double kf = 0x1.d3baeb0bee559p+30 * fexp2(fma(-0x1.bc56000000000p+21, irt, 0x1.0f5c280000000p+1 * lt));
    const double kb = 0x1.09b733934a1bap+26 * fexp2(fma(-0x1.30cab60000000p+26, irt, 0x1.4983fa0000000p+1 * lt));
    const double q = kf * C4 * C27 - kb * C28 * C26;
    cd4 -= q;
    cd26 += q;
    cd27 -= q;
    cd28 += q;
    }
    {  // R114 (elementary)
    const double kf = 0x1.bf08eb0000000p+32 * fexp2(fma(-0x1.febe000000000p+22, irt, 0.0 * lt));
    const double kb = 0x1.47e107e018af0p+30 * fexp2(fma(-0x1.dadb7c0000000p+25, irt, 0x1.f826680000000p-2 * lt));
    const double q = kf * C4 * C24 - kb * C28 * C22;
    cd4 -= q;
    cd22 += q;
    cd24 -= q;
    cd28 += q;
    }
    {  // R115 (elementary)
    const double kf = 0x1.efe9200000000p+26 * fexp2(fma(0x1.a042800000000p+22, irt, 0.0 * lt));
    const double kb = 0x1.41dc57b6679e3p+30 * fexp2(fma(-0x1.27309e2000000p+27, irt, -0x1.f587500000000p-3 * lt));
    const double q = kf * C6 * C6 - kb * C7 * C2;
    cd2 += q;
    cd6 = fma(-0x1.0000000000000p+1, q, cd6);
    cd7 += q;
    }
    {  // R116 (elementary)
    const double kf = 0x1.8727cda000000p+38 * fexp2(fma(-0x1.7f0e800000000p+25, irt, 0.0 * lt));
    const double kb = 0x1.fbbe360fde31fp+41 * fexp2(fma(-0x1.93f6522000000p+27, irt, -0x1.f587500000000p-3 * lt));
    const double q = kf * C6 * C6 - kb * C7 * C2;
    cd2 += q;
    cd6 = fma(-0x1.0000000000000p+1, q, cd6);
    cd7 += q;
    }
    {  // R117 (elementary)
    const double kf = 0x1.2a05f20000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.682ffb6cd52a6p+38 * fexp2(fma(-0x1.c5a7ae0000000p+28, irt, 0x1.ebca3e0000000p-9 * lt));
    const double q = kf * C6 * C10 - kb * C14 * C4;
    cd4 += q;
    cd6 -= q;
    cd10 -= q;
    cd14 += q;
    }
    {  // R118 (elementary)
    const double kf = 0x1.dcd6500000000p+29 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.9e6cbb7b0829ep+36 * fexp2(fma(-0x1.c4f8a40000000p+27, irt, -0x1.32263e0000000p-3 * lt));
    const double q = kf * C6 * C13 - kb * C15 * C2;
    cd2 += q;
    cd6 -= q;
    cd13 -= q;
    cd15 += q;
    }
    {  // R119 (elementary)
    const double kf = 0x1.19a1c74000000p+35 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.bfb78f5f12ffcp+37 * fexp2(fma(-0x1.93bb7a0000000p+26, irt, -0x1.32018a0000000p-3 * lt));
    const double q = kf * C6 * C13 - kb * C18 * C4;
    cd4 += q;
    cd6 -= q;
    cd13 -= q;
    cd18 += q;
    }
    {  // R120 (elementary)
    const double kf = 0x1.176592e000000p+37 * fexp2(fma(-0x1.78abbc0000000p+26, irt, 0.0 * lt));
    const double kb = 0x1.73bde0d44e40cp+42 * fexp2(fma(-0x1.53a8fc0000000p+28, irt, -0x1.0788120000000p-1 * lt));
    const double q = kf * C6 * C9 - kb * C16 * C4;
    cd4 += q;
    cd6 -= q;
    cd9 -= q;
    cd16 += q;
    }
    {  // R121 (elementary)
    const double kf = 0x1.5e00000000000p+30 * fexp2(fma(-0x1.7f0e800000000p+25, irt, 0x1.0000000000000p+1 * lt));
    const double kb = 0x1.015c47100e311p+28 * fexp2(fma(-0x1.65798c0000000p+25, irt, 0x1.d7ad6c0000000p+0 * lt));
    const double q = kf * C6 * C14 - kb * C7 * C11;
    cd6 -= q;
    cd7 += q;
    cd11 += q;
    cd14 -= q;
    }
    {  // R122 (elementary)
    const double kf = 0x1.b022388000000p+35 * fexp2(fma(-0x1.2630800000000p+21, irt, 0.0 * lt));
    const double kb = 0x1.354b3aaf5b64dp+36 * fexp2(fma(-0x1.14669c0000000p+29, irt, 0x1.7541100000000p-3 * lt));
    const double q = kf * C30 * C2 - kb * C9 * C1;
    cd1 += q;
    cd2 -= q;
    cd9 += q;
    cd30 -= q;
    }
    {  // R123 (elementary)
    const double kf = 0x1.74876e8000000p+35 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.8361a34217ff0p+40 * fexp2(fma(-0x1.387e500000000p+28, irt, -0x1.0280f20000000p+0 * lt));
    const double q = kf * C30 * C10 - kb * C20 * C3;
    cd3 += q;
    cd10 -= q;
    cd20 += q;
    cd30 -= q;
    }
    {  // R124 (elementary)
    const double kf = 0x1.74876e8000000p+35 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.8b9d30ee0c7d7p+42 * fexp2(fma(-0x1.909ab60000000p+28, irt, -0x1.1643aa0000000p+0 * lt));
    const double q = kf * C30 * C13 - kb * C21 * C3;
    cd3 += q;
    cd13 -= q;
    cd21 += q;
    cd30 -= q;
    }
    {  // R125 (elementary)
    const double kf = 0x1.f3ef17e000000p+35 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.d62a4c406fd3cp+36 * fexp2(fma(-0x1.2515fe0000000p+28, irt, -0x1.5486f00000000p-3 * lt));
    const double q = kf * C8 * C2 - kb * C11 * C1;
    cd1 += q;
    cd2 -= q;
    cd8 -= q;
    cd11 += q;
    }
    {  // R126 (elementary)
    const double kf = 0x1.9254d38000000p+36 * fexp2(fma(-0x1.8d18400000000p+23, irt, 0.0 * lt));
    const double kb = 0x1.081cab6f1a326p+38 * fexp2(fma(-0x1.9d56300000000p+20, irt, -0x1.2b7cbc0000000p-2 * lt));
    const double q = kf * C8 * C5 - kb * C10 * C3;
    cd3 += q;
    cd5 -= q;
    cd8 -= q;
    cd10 += q;
    }
    {  // R127 (elementary)
    const double kf = 0x1.5457af8000000p+32 * fexp2(fma(0x1.819ec00000000p+21, irt, 0.0 * lt));
    const double kb = 0x1.04c16aff0847ap+41 * fexp2(fma(-0x1.d9e3400000000p+27, irt, -0x1.e5377e0000000p-1 * lt));
    const double q = kf * C8 * C28 - kb * C14 * C3;
    cd3 += q;
    cd8 -= q;
    cd14 += q;
    cd28 -= q;
    }
    {  // R128 (elementary)
    const double kf = 0x1.2a05f20000000p+35 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.78f611f6c1ab5p+47 * fexp2(fma(-0x1.0586c60000000p+29, irt, -0x1.5f34d60000000p+0 * lt));
    const double q = kf * C8 * C10 - kb * C21 * C3;
    cd3 += q;
    cd8 -= q;
    cd10 -= q;
    cd21 += q;
    }
    {  // R129 (elementary)
    const double kf = 0x1.bf08eb0000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.45a6a9086658fp+41 * fexp2(fma(-0x1.b8ec060000000p+27, irt, -0x1.07e9100000000p+0 * lt));
    const double q = kf * C8 * C13 - kb * C23 * C3;
    cd3 += q;
    cd8 -= q;
    cd13 -= q;
    cd23 += q;
    }
    {  // R130 (elementary)
    const double kf = 0x1.bf08eb0000000p+35 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.04e7704893384p+43 * fexp2(fma(-0x1.e7648a0000000p+27, irt, -0x1.0154ca0000000p+0 * lt));
    const double q = kf * C8 * C15 - kb * C25 * C3;
    cd3 += q;
    cd8 -= q;
    cd15 -= q;
    cd25 += q;
    }
    {  // R132 (elementary)
    const double kf = 0x1.61e70f6000000p+37 * fexp2(fma(-0x1.f81ac80000000p+25, irt, 0.0 * lt));
    const double kb = 0x1.734bdec501c06p+32 * fexp2(fma(-0x1.40ed15b000000p+28, irt, 0x1.59d4300000000p-1 * lt));
    const double q = kf * C8 * C16 - kb * C9 * C11;
    cd8 -= q;
    cd9 += q;
    cd11 += q;
    cd16 -= q;
    }
    {  // R133 (elementary)
    const double kf = 0x1.6069972000000p+36 * fexp2(fma(0x1.070fc00000000p+21, irt, 0.0 * lt));
    const double kb = 0x1.0de7a343a17b7p+45 * fexp2(fma(-0x1.306a920000000p+28, irt, -0x1.5b20da0000000p+0 * lt));
    const double q = kf * C8 * C14 - kb * C24 * C3;
    cd3 += q;
    cd8 -= q;
    cd14 -= q;
    cd24 += q;
    }
    {  // R134 (elementary)
    const double kf = 0x1.74876e8000000p+35 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.24786e8a80cbfp+41 * fexp2(fma(-0x1.398c3c0000000p+29, irt, 0x1.03bf720000000p-3 * lt));
    const double q = kf * C8 * C22 - kb * C21 * C9;
    cd8 -= q;
    cd9 += q;
    cd21 += q;
    cd22 -= q;
    }
    {  // R135 (elementary)
    const double kf = 0x1.2a05f20000000p+32 * fexp2(fma(-0x1.7f0e800000000p+22, irt, 0.0 * lt));
    const double q = kf * C10 * C2;
    cd2 -= q;
    cd3 += q;
    cd4 += q;
    cd9 += q;
    cd10 -= q;
    }
    {  // R136 (elementary)
    const double kf = 0x1.f400000000000p+26 * fexp2(fma(-0x1.cd94100000000p+24, irt, 0x1.0000000000000p+1 * lt));
    const double kb = 0x1.0e859b1df9686p+31 * fexp2(fma(-0x1.d34da00000000p+25, irt, 0x1.7b0b3a0000000p+0 * lt));
    const double q = kf * C10 * C5 - kb * C13 * C3;
    cd3 += q;
    cd5 -= q;
    cd10 -= q;
    cd13 += q;
    }
    {  // R137 (elementary)
    const double kf = 0x1.74876e8000000p+40 * fexp2(fma(-0x1.7d45780000000p+25, irt, 0.0 * lt));
    const double kb = 0x1.66e74fdc11eefp+51 * fexp2(fma(-0x1.22c0d20000000p+29, irt, -0x1.1455860000000p+0 * lt));
    const double q = kf * C10 * C10 - kb * C21 * C5;
    cd5 += q;
    cd10 = fma(-0x1.0000000000000p+1, q, cd10);
    cd21 += q;
    }
    {  // R138 (elementary)
    const double kf = 0x1.2a05f20000000p+35 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.288f50f1a4e88p+47 * fexp2(fma(-0x1.0722820000000p+28, irt, -0x1.396bba0000000p+0 * lt));
    const double q = kf * C10 * C13 - kb * C25 * C3;
    cd3 += q;
    cd10 -= q;
    cd13 -= q;
    cd25 += q;
    }
    {  // R139 (elementary)
    const double kf = 0x1.3380000000000p+29 * fexp2(fma(-0x1.07fe080000000p+25, irt, 0x1.0000000000000p+1 * lt));
    const double kb = 0x1.29467677970c4p+27 * fexp2(fma(-0x1.af5b0e0000000p+25, irt, 0x1.fe00d20000000p+0 * lt));
    const double q = kf * C10 * C15 - kb * C13 * C13;
    cd10 -= q;
    cd13 = fma(0x1.0000000000000p+1, q, cd13);
    cd15 -= q;
    }
    {  // R141 (elementary)
    const double kf = 0x1.bf08eb0000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.4d3439b0c1360p+37 * fexp2(fma(-0x1.6cdcd00000000p+28, irt, 0x1.ed759e0000000p-3 * lt));
    const double q = kf * C10 * C22 - kb * C9 * C23;
    cd9 += q;
    cd10 -= q;
    cd22 -= q;
    cd23 += q;
    }
    {  // R142 (elementary)
    const double kf = 0x1.bf08eb0000000p+33 * fexp2(fma(-0x1.3265800000000p+21, irt, 0.0 * lt));
    const double kb = 0x1.b9fb5ac9f9a01p+32 * fexp2(fma(-0x1.2fbfbe0000000p+25, irt, -0x1.fe3fd60000000p-5 * lt));
    const double q = kf * C12 * C0 - kb * C0 * C10;
    cd10 += q;
    cd12 -= q;
    }
    {  // R143 (elementary)
    const double kf = 0x1.0c388d0000000p+33 * fexp2(fma(-0x1.3265800000000p+21, irt, 0.0 * lt));
    const double kb = 0x1.093069ac5137bp+32 * fexp2(fma(-0x1.2fbfbe0000000p+25, irt, -0x1.fe3fd60000000p-5 * lt));
    const double q = kf * C12 * C29 - kb * C29 * C10;
    cd10 += q;
    cd12 -= q;
    }
    {  // R144 (elementary)
    const double kf = 0x1.a13b860000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.d25ebdf246b74p+21 * fexp2(fma(-0x1.0d34e20000000p+28, irt, 0x1.0bd5dc0000000p-2 * lt));
    const double q = kf * C12 * C2 - kb * C9 * C4 * C3;
    cd2 -= q;
    cd3 += q;
    cd4 += q;
    cd9 += q;
    cd12 -= q;
    }
    {  // R145 (elementary)
    const double kf = 0x1.65a0bc0000000p+33 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.24514a881bd95p+34 * fexp2(fma(-0x1.7409700000000p+29, irt, 0x1.038fde0000000p-1 * lt));
    const double q = kf * C12 * C2 - kb * C28 * C9;
    cd2 -= q;
    cd9 += q;
    cd12 -= q;
    cd28 += q;
    }
    {  // R146 (elementary)
    const double kf = 0x1.04c533c000000p+36 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.16fd2b5de70a1p+39 * fexp2(fma(-0x1.048e7e0000000p+26, irt, -0x1.29cd600000000p-1 * lt));
    const double q = kf * C12 * C5 - kb * C3 * C13;
    cd3 += q;
    cd5 -= q;
    cd12 -= q;
    cd13 += q;
    }
    {  // R148 (elementary)
    const double kf = 0x1.bf08eb0000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.b9fb5ac9f9a01p+33 * fexp2(fma(-0x1.1c99660000000p+25, irt, -0x1.fe3fd60000000p-5 * lt));
    const double q = kf * C12 * C28 - kb * C28 * C10;
    cd10 += q;
    cd12 -= q;
    }
    {  // R149 (elementary)
    const double kf = 0x1.65a0bc0000000p+33 * fexp2(fma(0x1.2323400000000p+21, irt, 0.0 * lt));
    const double kb = 0x1.5fdcfbc749bcap+44 * fexp2(fma(-0x1.286f680000000p+28, irt, -0x1.495d4e0000000p+0 * lt));
    const double q = kf * C12 * C13 - kb * C25 * C3;
    cd3 += q;
    cd12 -= q;
    cd13 -= q;
    cd25 += q;
    }
    {  // R150 (elementary)
    const double kf = 0x1.dcd6500000000p+33 * fexp2(fma(0x1.2323400000000p+21, irt, 0.0 * lt));
    const double kb = 0x1.c7c6a03d0c843p+30 * fexp2(fma(-0x1.b1c4380000000p+25, irt, -0x1.1f11080000000p-4 * lt));
    const double q = kf * C12 * C15 - kb * C13 * C13;
    cd12 -= q;
    cd13 = fma(0x1.0000000000000p+1, q, cd13);
    cd15 -= q;
    }
    {  // R151 (elementary)
    const double kf = 0x1.0c388d0000000p+33 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.093069ac5137bp+32 * fexp2(fma(-0x1.1c99660000000p+25, irt, -0x1.fe3fd60000000p-5 * lt));
    const double q = kf * C12 * C9 - kb * C9 * C10;
    cd10 += q;
    cd12 -= q;
    }
    {  // R152 (elementary)
    const double kf = 0x1.a13b860000000p+32 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.9c84329a494e9p+31 * fexp2(fma(-0x1.1c99660000000p+25, irt, -0x1.fe3fd60000000p-5 * lt));
    const double q = kf * C12 * C16 - kb * C16 * C10;
    cd10 += q;
    cd12 -= q;
    }
    {  // R153 (elementary)
    const double kf = 0x1.a13b860000000p+33 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.76b6e44aca862p+31 * fexp2(fma(-0x1.e7799a0000000p+27, irt, 0x1.d31fce0000000p-2 * lt));
    const double q = kf * C12 * C16 - kb * C14 * C9;
    cd9 += q;
    cd12 -= q;
    cd14 += q;
    cd16 -= q;
    }
    {  // R154 (elementary)
    const double kf = 0x1.2a05f20000000p+35 * fexp2(fma(0x1.18e2400000000p+21, irt, 0.0 * lt));
    const double kb = 0x1.f69f3d1f889f8p+30 * fexp2(fma(-0x1.27546c0000000p+26, irt, -0x1.700fc80000000p-6 * lt));
    const double q = kf * C12 * C27 - kb * C26 * C13;
    cd12 -= q;
    cd13 += q;
    cd26 += q;
    cd27 -= q;
    }
    {  // R155 (elementary)
    const double kf = 0x1.093d9c8000000p+35 * fexp2(fma(-0x1.e67b100000000p+26, irt, 0.0 * lt));
    const double kb = 0x1.1c14d4cf886bap+38 * fexp2(fma(-0x1.877ada0000000p+23, irt, -0x1.e7dc7a0000000p-2 * lt));
    const double q = kf * C13 * C2 - kb * C18 * C1;
    cd1 += q;
    cd2 -= q;
    cd13 -= q;
    cd18 += q;
    }
    {  // R156 (elementary)
    const double kf = 0x1.135f9b0000000p+31 * fexp2(fma(-0x1.443ddc0000000p+26, irt, 0.0 * lt));
    const double kb = 0x1.8c19d104f8309p+30 * fexp2(fma(-0x1.1f4f320000000p+28, irt, 0x1.49cdc40000000p-3 * lt));
    const double q = kf * C13 * C2 - kb * C14 * C4;
    cd2 -= q;
    cd4 += q;
    cd13 -= q;
    cd14 += q;
    }
    {  // R157 (elementary)
    const double kf = 0x1.cbc05a94b7ae3p+26 * fexp2(fma(-0x1.4ab4280000000p+24, irt, 0x1.3c28f60000000p+1 * lt));
    const double kb = 0x1.33d32b8d72070p+30 * fexp2(fma(-0x1.7438ec0000000p+26, irt, 0x1.485f060000000p+1 * lt));
    const double q = kf * C13 * C7 - kb * C15 * C6;
    cd6 += q;
    cd7 -= q;
    cd13 -= q;
    cd15 += q;
    }
    {  // R159 (elementary)
    const double kf = 0x1.7c64c3796fee8p+33 * fexp2(fma(-0x1.525d180000000p+25, irt, 0x1.99999a0000000p-4 * lt));
    const double kb = 0x1.272996025235ep+40 * fexp2(fma(-0x1.ca88ba0000000p+22, irt, -0x1.1394da0000000p+0 * lt));
    const double q = kf * C13 * C13 - kb * C26 * C3;
    cd3 += q;
    cd13 = fma(-0x1.0000000000000p+1, q, cd13);
    cd26 += q;
    }
    {  // R160 (elementary)
    const double kf = 0x1.8a952f0000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.71f4a2db6b13fp+41 * fexp2(fma(-0x1.66f20c0000000p+28, irt, 0x1.2466620000000p-4 * lt));
    const double q = kf * C13 * C11 - kb * C9 * C15;
    cd9 += q;
    cd11 -= q;
    cd13 -= q;
    cd15 += q;
    }
    {  // R161 (elementary)
    const double kf = 0x1.03c958f262512p+27 * fexp2(fma(-0x1.761d700000000p+24, irt, 0x1.67ae140000000p+1 * lt));
    const double kb = 0x1.ff99f344c769fp+27 * fexp2(fma(-0x1.7248c40000000p+26, irt, 0x1.5fbadc0000000p+1 * lt));
    const double q = kf * C13 * C14 - kb * C15 * C11;
    cd11 += q;
    cd13 -= q;
    cd14 -= q;
    cd15 += q;
    }
    {  // R162 (elementary)
    const double kf = 0x1.4b74d0516bc5fp+28 * fexp2(fma(-0x1.3d4c840000000p+25, irt, 0x1.8000000000000p+0 * lt));
    const double kb = 0x1.4b3cc1ba18aa8p+29 * fexp2(fma(-0x1.29ab5e0000000p+26, irt, 0x1.330fd00000000p+0 * lt));
    const double q = kf * C13 * C19 - kb * C15 * C17;
    cd13 -= q;
    cd15 += q;
    cd17 += q;
    cd19 -= q;
    }
    {  // R163 (elementary)
    const double kf = 0x1.b9f115c1e507fp+26 * fexp2(fma(-0x1.3d4c840000000p+25, irt, 0x1.8000000000000p+0 * lt));
    const double kb = 0x1.60ed67d6c7876p+31 * fexp2(fma(-0x1.79b10c0000000p+25, irt, 0x1.422f060000000p+0 * lt));
    const double q = kf * C13 * C19 - kb * C15 * C18;
    cd13 -= q;
    cd15 += q;
    cd18 += q;
    cd19 -= q;
    }
    {  // R164 (elementary)
    const double kf = 0x1.c600000000000p+25 * fexp2(fma(-0x1.25ada40000000p+25, irt, 0x1.0000000000000p+1 * lt));
    const double kb = 0x1.1b59d46c6e2f7p+25 * fexp2(fma(-0x1.af2e600000000p+23, irt, 0x1.f96c620000000p+0 * lt));
    const double q = kf * C13 * C25 - kb * C15 * C23;
    cd13 -= q;
    cd15 += q;
    cd23 += q;
    cd25 -= q;
    }
    {  // R165 (elementary)
    const double kf = 0x1.2f2da9c097388p+28 * fexp2(fma(-0x1.4d947c0000000p+25, irt, 0x1.bd70a40000000p+0 * lt));
    const double kb = 0x1.0b78db3c2772ep+27 * fexp2(fma(-0x1.e9d50a0000000p+25, irt, 0x1.c9a1760000000p+0 * lt));
    const double q = kf * C13 * C27 - kb * C15 * C26;
    cd13 -= q;
    cd15 += q;
    cd26 += q;
    cd27 -= q;
    }
    {  // R166 (elementary)
    const double kf = 0x1.550f7dca70000p+41 * fexp2(fma(-0x1.0f54f00000000p+26, irt, -0x1.0000000000000p+0 * lt));
    const double kb = 0x1.199834ce95c1bp+31 * fexp2(fma(-0x1.46cef00000000p+22, irt, -0x1.88d9fa0000000p-1 * lt));
    const double q = kf * C11 * C28 - kb * C28 * C9 * C3;
    cd3 += q;
    cd9 += q;
    cd11 -= q;
    }
    {  // R168 (elementary)
    const double kf = 0x1.90d75b4000000p+33 * fexp2(fma(-0x1.98b1000000000p+20, irt, 0.0 * lt));
    const double kb = 0x1.b06baf6d5802cp+33 * fexp2(fma(-0x1.0c1cd60000000p+27, irt, 0x1.c459100000000p-3 * lt));
    const double q = kf * C11 * C2 - kb * C9 * C6;
    cd2 -= q;
    cd6 += q;
    cd9 += q;
    cd11 -= q;
    }
    {  // R169 (elementary)
    const double kf = 0x1.0c388d0000000p+34 * fexp2(fma(-0x1.cbb7800000000p+21, irt, 0.0 * lt));
    const double kb = 0x1.83e283b304326p+34 * fexp2(fma(-0x1.46ce560000000p+26, irt, 0x1.7a658c0000000p-2 * lt));
    const double q = kf * C17 * C2 - kb * C14 * C6;
    cd2 -= q;
    cd6 += q;
    cd14 += q;
    cd17 -= q;
    }
    {  // R170 (elementary)
    const double kf = 0x1.458e3fdf782b8p+17 * fexp2(fma(0x1.c2bea00000000p+23, irt, 0x1.e666660000000p+2 * lt));
    const double kb = 0x1.268fdb1780c20p+14 * fexp2(fma(-0x1.6ceb9c0000000p+26, irt, 0x1.fa44d00000000p+2 * lt));
    const double q = kf * C18 * C2 - kb * C14 * C6;
    cd2 -= q;
    cd6 += q;
    cd14 += q;
    cd18 -= q;
    }
    {  // R171 (elementary)
    const double kf = 0x1.2a05f20000000p+33 * fexp2(fma(0x1.819ec00000000p+21, irt, 0.0 * lt));
    const double kb = 0x1.22320c06e8519p+32 * fexp2(fma(-0x1.2c4e140000000p+29, irt, 0x1.b157ac0000000p-1 * lt));
    const double q = kf * C20 * C2 - kb * C9 * C11;
    cd2 -= q;
    cd9 += q;
    cd11 += q;
    cd20 -= q;
    }
    {  // R172 (elementary)
    const double kf = 0x1.d073d9cf0fbdap+33 * fexp2(fma(-0x1.fcf8e00000000p+22, irt, 0x1.cccccc0000000p-1 * lt));
    const double kb = 0x1.00a5a07be73f2p+40 * fexp2(fma(-0x1.f682f20000000p+26, irt, 0x1.36be7a0000000p-2 * lt));
    const double q = kf * C20 * C5 - kb * C21 * C3;
    cd3 += q;
    cd5 -= q;
    cd20 -= q;
    cd21 += q;
    }
    {  // R173 (elementary)
    const double kf = 0x1.d4040197c6493p+32 * fexp2(fma(-0x1.0337600000000p+22, irt, -0x1.63d70a0000000p+0 * lt));
    const double kb = 0x1.c0f04012184b9p+31 * fexp2(fma(-0x1.602dbc0000000p+28, irt, -0x1.9a2ec20000000p-1 * lt));
    const double q = kf * C23 * C2 - kb * C14 * C11;
    cd2 -= q;
    cd11 += q;
    cd14 += q;
    cd23 -= q;
    }
    {  // R175 (elementary)
    const double kf = 0x1.908b100000000p+29 * fexp2(fma(-0x1.eec8100000000p+23, irt, 0.0 * lt));
    const double kb = 0x1.31aca5a80662ep+30 * fexp2(fma(-0x1.0949440000000p+26, irt, 0x1.c068dc0000000p-4 * lt));
    const double q = kf * C26 * C2 - kb * C25 * C6;
    cd2 -= q;
    cd6 += q;
    cd25 += q;
    cd26 -= q;
    }
    {  // R176 (elementary)
    const double kf = 0x1.7d78400000000p+31 * fexp2(fma(-0x1.b428400000000p+21, irt, 0.0 * lt));
    const double kb = 0x1.0bb1ef703d708p+13 * fexp2(fma(-0x1.5514f40000000p+28, irt, 0x1.d2949a0000000p+0 * lt));
    const double q = kf * C22 * C2 - kb * C9 * C9 * C4;
    cd2 -= q;
    cd4 += q;
    cd9 = fma(0x1.0000000000000p+1, q, cd9);
    cd22 -= q;
    }
    {  // R177 (elementary)
    const double kf = 0x1.2a05f20000000p+33 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.b422b03570c62p+19 * fexp2(fma(-0x1.48e7980000000p+28, irt, 0x1.915b580000000p+0 * lt));
    const double q = kf * C22 * C22 - kb * C21 * C9 * C9;
    cd9 = fma(0x1.0000000000000p+1, q, cd9);
    cd21 += q;
    cd22 = fma(-0x1.0000000000000p+1, q, cd22);
    }
    {  // R284 (elementary)
    const double kf = 0x1.f62b4c4000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C1 * C13;
    cd1 -= q;
    cd3 += q;
    cd5 += q;
    cd9 += q;
    cd13 -= q;
    }
    {  // R285 (elementary)
    const double kf = 0x1.2201e32a77f7bp+29 * fexp2(fma(-0x1.c138000000000p+19, irt, 0x1.d47ae20000000p+0 * lt));
    const double kb = 0x1.3e062d8615213p+28 * fexp2(fma(-0x1.bf73c40000000p+25, irt, 0x1.6795d40000000p+0 * lt));
    const double q = kf * C1 * C25 - kb * C32 * C3;
    cd1 -= q;
    cd3 += q;
    cd25 -= q;
    cd32 += q;
    }
    {  // R286 (elementary)
    const double kf = 0x1.984ab48000000p+36 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.11eac82e156a4p+42 * fexp2(fma(-0x1.2e77ea0000000p+28, irt, -0x1.0696c40000000p-1 * lt));
    const double q = kf * C1 * C26 - kb * C33 * C3;
    cd1 -= q;
    cd3 += q;
    cd26 -= q;
    cd33 += q;
    }
    {  // R287 (elementary)
    const double kf = 0x1.2309ce5400000p+42 * fexp2(fma(-0x1.1499920000000p+26, irt, 0.0 * lt));
    const double kb = 0x1.45c4e91a8cbc0p+45 * fexp2(fma(-0x1.5cd4a60000000p+28, irt, 0x1.0769660000000p-2 * lt));
    const double q = kf * C4 * C6 - kb * C28 * C2;
    cd2 += q;
    cd4 -= q;
    cd6 -= q;
    cd28 += q;
    }
    {  // R288 (elementary)
    const double kf = 0x1.594458ff7aee3p+27 * fexp2(fma(0x1.c02e600000000p+22, irt, 0x1.0000000000000p-1 * lt));
    const double q = kf * C4 * C13;
    cd4 -= q;
    cd5 += q;
    cd13 -= q;
    cd14 += q;
    }
    {  // R290 (elementary)
    const double kf = 0x1.59b4fa0000000p+32 * fexp2(fma(-0x1.7f0e800000000p+22, irt, 0.0 * lt));
    const double q = kf * C10 * C2;
    cd2 -= q;
    cd3 = fma(0x1.0000000000000p+1, q, cd3);
    cd10 -= q;
    cd16 += q;
    }
    {  // R291 (elementary)
    const double kf = 0x1.1e1a300000000p+31 * fexp2(fma(-0x1.7f0e800000000p+22, irt, 0.0 * lt));
    const double kb = 0x1.d1eb495f65ab8p+35 * fexp2(fma(-0x1.f2a4360000000p+27, irt, -0x1.4b04260000000p-2 * lt));
    const double q = kf * C10 * C2 - kb * C14 * C1;
    cd1 += q;
    cd2 -= q;
    cd10 -= q;
    cd14 += q;
    }
    {  // R292 (elementary)
    const double kf = 0x1.74876e8000000p+37 * fexp2(fma(-0x1.5ec8c80000000p+25, irt, 0.0 * lt));
    const double q = kf * C10 * C10;
    cd3 = fma(0x1.0000000000000p+1, q, cd3);
    cd10 = fma(-0x1.0000000000000p+1, q, cd10);
    cd21 += q;
    }
    {  // R293 (elementary)
    const double kf = 0x1.35630d4f905a4p+28 * fexp2(fma(0x1.dd8a000000000p+21, irt, 0x1.0000000000000p-2 * lt));
    const double q = kf * C12 * C28;
    cd5 += q;
    cd12 -= q;
    cd14 += q;
    cd28 -= q;
    }
    {  // R294 (elementary)
    const double kf = 0x1.b9086c43db9e3p+30 * fexp2(fma(-0x1.6760000000000p+15, irt, 0x1.28f5c20000000p-2 * lt));
    const double kb = 0x1.b730e2956b21bp+32 * fexp2(fma(-0x1.93eb4e0000000p+24, irt, -0x1.31ed9e0000000p-3 * lt));
    const double q = kf * C23 * C2 - kb * C32 * C1;
    cd1 += q;
    cd2 -= q;
    cd23 -= q;
    cd32 += q;
    }
    {  // R295 (elementary)
    const double kf = 0x1.d56f8cc313341p+24 * fexp2(fma(0x1.8855800000000p+20, irt, 0x1.9c28f60000000p+0 * lt));
    const double kb = 0x1.e5090f02eb8fdp+25 * fexp2(fma(-0x1.ad39fc0000000p+25, irt, 0x1.6d20b00000000p+0 * lt));
    const double q = kf * C23 * C2 - kb * C21 * C6;
    cd2 -= q;
    cd6 += q;
    cd21 += q;
    cd23 -= q;
    }
    {  // R296 (elementary)
    const double kf = 0x1.5c17540000000p+31 * fexp2(fma(-0x1.cdbb200000000p+22, irt, 0.0 * lt));
    const double kb = 0x1.423f4502b72a5p+25 * fexp2(fma(-0x1.4faba20000000p+24, irt, 0x1.0c475e0000000p-1 * lt));
    const double q = kf * C1 * C33 - kb * C32 * C4;
    cd1 -= q;
    cd4 += q;
    cd32 += q;
    cd33 -= q;
    }
    {  // R297 (elementary)
    const double kf = 0x1.5c17540000000p+31 * fexp2(fma(-0x1.cdbb200000000p+22, irt, 0.0 * lt));
    const double q = kf * C1 * C33;
    cd1 -= q;
    cd4 += q;
    cd9 += q;
    cd13 += q;
    cd33 -= q;
    }
    {  // R298 (elementary)
    const double kf = 0x1.c086634000000p+34 * fexp2(fma(-0x1.386e6c0000000p+27, irt, 0.0 * lt));
    const double q = kf * C2 * C33;
    cd2 -= q;
    cd6 += q;
    cd9 += q;
    cd13 += q;
    cd33 -= q;
    }
    {  // R299 (elementary)
    const double kf = 0x1.537b72566356bp+31 * fexp2(fma(-0x1.3319300000000p+23, irt, 0x1.28f5c20000000p+0 * lt));
    const double kb = 0x1.48d3303026ff9p+26 * fexp2(fma(-0x1.ee24b00000000p+24, irt, 0x1.b813aa0000000p+0 * lt));
    const double q = kf * C3 * C33 - kb * C5 * C32;
    cd3 -= q;
    cd5 += q;
    cd32 += q;
    cd33 -= q;
    }
    {  // R300 (elementary)
    const double kf = 0x1.537b72566356bp+31 * fexp2(fma(-0x1.3319300000000p+23, irt, 0x1.28f5c20000000p+0 * lt));
    const double q = kf * C3 * C33;
    cd3 -= q;
    cd5 += q;
    cd9 += q;
    cd13 += q;
    cd33 -= q;
    }
    {  // R301 (elementary)
    const double kf = 0x1.095e5bb3014a1p+31 * fexp2(fma(0x1.1c3da00000000p+22, irt, 0x1.75c2900000000p-1 * lt));
    const double q = kf * C4 * C33;
    cd4 -= q;
    cd9 += q;
    cd13 += q;
    cd28 += q;
    cd33 -= q;
    }
    {  // R302 (elementary)
    const double kf = 0x1.66d1e90000000p+31 * fexp2(fma(-0x1.7c99980000000p+25, irt, 0.0 * lt));
    const double q = kf * C6 * C33;
    cd6 -= q;
    cd7 += q;
    cd9 += q;
    cd13 += q;
    cd33 -= q;
    }
    {  // R303 (elementary)
    const double kf = 0x1.43e599fad54a0p+27 * fexp2(fma(-0x1.79f1e80000000p+24, irt, 0x1.c51eb80000000p+0 * lt));
    const double q = kf * C13 * C33;
    cd9 += q;
    cd15 += q;
    cd33 -= q;
    }
    {  // R305 (elementary)
    const double kf = 0x1.176592e000000p+37 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C1 * C32;
    cd1 -= q;
    cd3 += q;
    cd10 += q;
    cd16 += q;
    cd32 -= q;
    }
    {  // R306 (elementary)
    const double kf = 0x1.142f200000000p+24 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C2 * C32;
    cd2 -= q;
    cd4 += q;
    cd9 += q;
    cd14 += q;
    cd32 -= q;
    }
    {  // R307 (elementary)
    const double kf = 0x1.6694e00000000p+24 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C2 * C32;
    cd2 -= q;
    cd4 += q;
    cd11 = fma(0x1.0000000000000p+1, q, cd11);
    cd32 -= q;
    }
    {  // R308 (elementary)
    const double kf = 0x1.47d3570000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.a8fb8237c1f7fp+26 * fexp2(fma(-0x1.7b64040000000p+25, irt, 0x1.4dd2f20000000p+0 * lt));
    const double q = kf * C3 * C32 - kb * C11 * C13;
    cd3 -= q;
    cd11 += q;
    cd13 += q;
    cd32 -= q;
    }
    {  // R309 (elementary)
    const double kf = 0x1.47d3570000000p+33 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.046dd72d54b5cp+34 * fexp2(fma(-0x1.1294a40000000p+28, irt, 0x1.3ddace0000000p-2 * lt));
    const double q = kf * C3 * C32 - kb * C5 * C24;
    cd3 -= q;
    cd5 += q;
    cd24 += q;
    cd32 -= q;
    }
    {  // R310 (elementary)
    const double kf = 0x1.65a0bc0000000p+33 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.998dc7b338cb7p+36 * fexp2(fma(-0x1.506b660000000p+28, irt, 0x1.a501e20000000p-3 * lt));
    const double q = kf * C4 * C32 - kb * C24 * C28;
    cd4 -= q;
    cd24 += q;
    cd28 += q;
    cd32 -= q;
    }
    {  // R311 (elementary)
    const double kf = 0x1.c086634000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.928f8da4a0109p+31 * fexp2(fma(-0x1.13fb980000000p+25, irt, 0x1.53a9f40000000p-2 * lt));
    const double q = kf * C4 * C32 - kb * C17 * C11;
    cd4 -= q;
    cd11 += q;
    cd17 += q;
    cd32 -= q;
    }
    {  // R313 (elementary)
    const double kf = 0x1.a37ad63ee0d7ap+31 * fexp2(fma(-0x1.da7cc00000000p+23, irt, 0x1.570a3e0000000p+1 * lt));
    const double kb = 0x1.07331e88d6a71p+23 * fexp2(fma(-0x1.05b2000000000p+24, irt, 0x1.9be4ce0000000p+1 * lt));
    const double q = kf * C1 * C34 - kb * C35 * C4;
    cd1 -= q;
    cd4 += q;
    cd34 -= q;
    cd35 += q;
    }
    {  // R314 (elementary)
    const double kf = 0x1.2b7b3332f7afep+33 * fexp2(fma(-0x1.af51f80000000p+24, irt, 0x1.451eb80000000p+1 * lt));
    const double kb = 0x1.89372542cb634p+25 * fexp2(fma(-0x1.20106a0000000p+25, irt, 0x1.8e76740000000p+1 * lt));
    const double q = kf * C3 * C34 - kb * C5 * C35;
    cd3 -= q;
    cd5 += q;
    cd34 -= q;
    cd35 += q;
    }
    {  // R315 (elementary)
    const double kf = 0x1.1b95b6e591453p+31 * fexp2(fma(-0x1.dd0d000000000p+21, irt, 0x1.cccccc0000000p+0 * lt));
    const double kb = 0x1.0c5eb268218f8p+26 * fexp2(fma(-0x1.2a77280000000p+26, irt, 0x1.2252be0000000p+1 * lt));
    const double q = kf * C4 * C34 - kb * C28 * C35;
    cd4 -= q;
    cd28 += q;
    cd34 -= q;
    cd35 += q;
    }
    {  // R316 (elementary)
    const double kf = 0x1.0deee377d84c4p+23 * fexp2(fma(-0x1.7f0e800000000p+22, irt, 0x1.5c28f60000000p+1 * lt));
    const double kb = 0x1.ebe96a4a3214ap+27 * fexp2(fma(-0x1.e56b940000000p+25, irt, 0x1.6082160000000p+1 * lt));
    const double q = kf * C35 * C7 - kb * C34 * C6;
    cd6 += q;
    cd7 -= q;
    cd34 += q;
    cd35 -= q;
    }
    {  // R317 (elementary)
    const double kf = 0x1.aaae5dea71f54p+22 * fexp2(fma(-0x1.c8b9e00000000p+24, irt, 0x1.d333340000000p+1 * lt));
    const double kb = 0x1.39886c0c018d4p+21 * fexp2(fma(-0x1.71eaf00000000p+25, irt, 0x1.db10240000000p+1 * lt));
    const double q = kf * C13 * C34 - kb * C15 * C35;
    cd13 -= q;
    cd15 += q;
    cd34 -= q;
    cd35 += q;
    }
    {  // R319 (elementary)
    const double kf = 0x1.671e344000000p+36 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.12f40280315c3p+33 * fexp2(fma(-0x1.41453c0000000p+28, irt, 0x1.4343960000000p+0 * lt));
    const double q = kf * C1 * C35 - kb * C14 * C26;
    cd1 -= q;
    cd14 += q;
    cd26 += q;
    cd35 -= q;
    }
    {  // R321 (elementary)
    const double kf = 0x1.9f15df95c4c12p+31 * fexp2(fma(-0x1.c697000000000p+21, irt, 0x1.1851ec0000000p+1 * lt));
    const double kb = 0x1.abb4bd9906c0fp+23 * fexp2(fma(-0x1.8a8c2e0000000p+25, irt, 0x1.dd3fd00000000p+1 * lt));
    const double q = kf * C3 * C35 - kb * C26 * C13;
    cd3 -= q;
    cd13 += q;
    cd26 += q;
    cd35 -= q;
    }
    {  // R322 (elementary)
    const double kf = 0x1.671e344000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.002eff50b142bp+31 * fexp2(fma(-0x1.06ba520000000p+25, irt, 0x1.21e6260000000p-1 * lt));
    const double q = kf * C4 * C35 - kb * C17 * C26;
    cd4 -= q;
    cd17 += q;
    cd26 += q;
    cd35 -= q;
    }
    {  // R323 (elementary)
    const double kf = 0x1.dd613dfd44cf7p+26 * fexp2(fma(0x1.e1b0800000000p+21, irt, 0x1.051eb80000000p-2 * lt));
    const double kb = 0x1.1a520bbe51107p+35 * fexp2(fma(-0x1.9a0e620000000p+27, irt, 0x1.692a660000000p-5 * lt));
    const double q = kf * C6 * C35 - kb * C34 * C2;
    cd2 += q;
    cd6 -= q;
    cd34 += q;
    cd35 -= q;
    }
    {  // R324 (elementary)
    const double kf = 0x1.671e344000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C6 * C35;
    cd4 += q;
    cd6 -= q;
    cd14 += q;
    cd26 += q;
    cd35 -= q;
    }
    {  // R325 (elementary)
    const double kf = 0x1.380d0819d1fcap+31 * fexp2(fma(0.0, irt, -0x1.47ae140000000p-2 * lt));
    const double kb = 0x1.f2fec18bd14e8p+29 * fexp2(fma(-0x1.545af20000000p+23, irt, 0x1.583de40000000p-5 * lt));
    const double q = kf * C13 * C35 - kb * C26 * C26;
    cd13 -= q;
    cd26 = fma(0x1.0000000000000p+1, q, cd26);
    cd35 -= q;
    }
    {  // R1 (third_body)
    const double kf = 0x1.bf08eb0000000p+27 * fexp2(fma(0.0, irt, -0x1.0000000000000p+0 * lt));
    const double kb = 0x1.bfd6620e8f8eap+42 * fexp2(fma(-0x1.dac2b02000000p+28, irt, -0x1.1f23240000000p+0 * lt));
    const double q = (kf * C1 * C1 - kb * C2) * M0();
    cd1 = fma(-0x1.0000000000000p+1, q, cd1);
    cd2 += q;
    }
    {  // R2 (third_body)
    const double kf = 0x1.d1a94a2000000p+29 * fexp2(fma(0.0, irt, -0x1.0000000000000p+0 * lt));
    const double kb = 0x1.c38c12b09edefp+39 * fexp2(fma(-0x1.9581860000000p+28, irt, -0x1.5ea1c60000000p-1 * lt));
    const double q = (kf * C1 * C3 - kb * C4) * M1();
    cd1 -= q;
    cd3 -= q;
    cd4 += q;
    }
    {  // R12 (falloff)
    const double kinf_f = 0x1.12a8800000000p+24 * fexp2(fma(-0x1.3088f00000000p+23, irt, 0.0 * lt));
    const double k0_f = 0x1.1f0e540000000p+29 * fexp2(fma(-0x1.7f0e800000000p+23, irt, 0.0 * lt));
    const double kinf_b = 0x1.ed4d6401a2176p+44 * fexp2(fma(-0x1.03b99c5000000p+29, irt, -0x1.ed3bb00000000p-1 * lt));
    const double k0_b = 0x1.01c8e2ed6e16dp+50 * fexp2(fma(-0x1.04f3b29000000p+29, irt, -0x1.ed3bb00000000p-1 * lt));
    const double m_ = M2();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    const double pr_f = k0_f * conc / fmax(kinf_f, 1.0e-60);
    const double kf = kinf_f * pr_f / (1.0 + pr_f);
    const double pr_b = k0_b * conc / fmax(kinf_b, 1.0e-60);
    const double kb = kinf_b * pr_b / (1.0 + pr_b);
    const double q = kf * C1 * C9 - kb * C16;
    cd1 -= q;
    cd9 -= q;
    cd16 += q;
    }
    {  // R33 (third_body)
    const double kf = 0x1.865566a97a645p+33 * fexp2(fma(0.0, irt, -0x1.b851ec0000000p-1 * lt));
    const double kb = 0x1.fe0218b17dae9p+43 * fexp2(fma(-0x1.865f740000000p+27, irt, -0x1.be61ae0000000p-1 * lt));
    const double q = (kf * C3 * C2 - kb * C6) * M3();
    cd2 -= q;
    cd3 -= q;
    cd6 += q;
    }
    {  // R39 (third_body)
    const double kf = 0x1.d1a94a2000000p+30 * fexp2(fma(0.0, irt, -0x1.0000000000000p+0 * lt));
    const double kb = 0x1.d86f04f01afeep+41 * fexp2(fma(-0x1.9d073a0000000p+28, irt, -0x1.4cae000000000p-1 * lt));
    const double q = (kf * C3 * C3 - kb * C5) * M4();
    cd3 = fma(-0x1.0000000000000p+1, q, cd3);
    cd5 += q;
    }
    {  // R43 (third_body)
    const double kf = 0x1.38a388a43c000p+36 * fexp2(fma(0.0, irt, -0x1.0000000000000p+1 * lt));
    const double kb = 0x1.c93e0a5a9fea7p+49 * fexp2(fma(-0x1.daddfc0000000p+28, irt, -0x1.c12d780000000p+0 * lt));
    const double q = (kf * C3 * C4 - kb * C28) * M5();
    cd3 -= q;
    cd4 -= q;
    cd28 += q;
    }
    {  // R50 (falloff)
    const double kinf_f = 0x1.176592e000000p+39 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double k0_f = 0x1.9324709d7b3d5p+41 * fexp2(fma(-0x1.9891c00000000p+22, irt, -0x1.6147ae0000000p+1 * lt));
    const double kinf_b = 0x1.32bb872223823p+54 * fexp2(fma(-0x1.ba97ac0000000p+28, irt, -0x1.5a5d280000000p-3 * lt));
    const double k0_b = 0x1.ba97deee93036p+56 * fexp2(fma(-0x1.c0f9f40000000p+28, irt, -0x1.76ed680000000p+1 * lt));
    const double m_ = M6();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.c083120000000p-2, fexp2(-(0x1.03bf9f2c1c437p-6 * T)), fc);
    fc = fma(0x1.1fbe760000000p-1, fexp2(-(0x1.0336e4addcb01p-12 * T)), fc);
    fc = fma(0x1.0000000000000p+0, fexp2(-(0x1.818f6c85dac80p+13 * invT)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C3 * C10 - kb * C13;
    cd3 -= q;
    cd10 -= q;
    cd13 += q;
    }
    {  // R52 (falloff)
    const double kinf_f = 0x1.cec504d9ae2dfp+38 * fexp2(fma(-0x1.11cdc00000000p+21, irt, -0x1.1168720000000p-1 * lt));
    const double k0_f = 0x1.2eacabe244721p+48 * fexp2(fma(-0x1.378dd00000000p+23, irt, -0x1.30a3d80000000p+2 * lt));
    const double kinf_b = 0x1.06c1c5b7c65cap+56 * fexp2(fma(-0x1.a7cfa79000000p+28, irt, -0x1.6401a40000000p-1 * lt));
    const double k0_b = 0x1.57b3c8733ba72p+65 * fexp2(fma(-0x1.af687a9000000p+28, irt, -0x1.3af7120000000p+2 * lt));
    const double m_ = M7();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.bc6a7e0000000p-3, fexp2(-(0x1.3f6ba49a91758p-6 * T)), fc);
    fc = fma(0x1.90e5600000000p-1, fexp2(-(0x1.012fef8327e8fp-11 * T)), fc);
    fc = fma(0x1.0000000000000p+0, fexp2(-(0x1.39f76d1611d3bp+13 * invT)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C3 * C13 - kb * C15;
    cd3 -= q;
    cd13 -= q;
    cd15 += q;
    }
    {  // R54 (falloff)
    const double kinf_f = 0x1.4469543cee0f0p+34 * fexp2(fma(0x1.09a0000000000p+20, irt, 0x1.eb851e0000000p-2 * lt));
    const double k0_f = 0x1.f530f43ca09eap+37 * fexp2(fma(-0x1.b215000000000p+20, irt, -0x1.48f5c20000000p+1 * lt));
    const double kinf_b = 0x1.7620ae93a1631p+50 * fexp2(fma(-0x1.5f72120000000p+28, irt, 0x1.85eb740000000p-2 * lt));
    const double k0_b = 0x1.20ff6565d9665p+54 * fexp2(fma(-0x1.622dc60000000p+28, irt, -0x1.55a9000000000p+1 * lt));
    const double m_ = M8();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.bda5120000000p-3, fexp2(-(0x1.5ce327092e76fp-8 * T)), fc);
    fc = fma(0x1.9096bc0000000p-1, fexp2(-(0x1.128d07060469dp-11 * T)), fc);
    fc = fma(0x1.0000000000000p+0, fexp2(-(0x1.28340d253757ep+13 * invT)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C3 * C11 - kb * C14;
    cd3 -= q;
    cd11 -= q;
    cd14 += q;
    }
    {  // R56 (falloff)
    const double kinf_f = 0x1.114edc398b4b1p+33 * fexp2(fma(-0x1.cba7e00000000p+23, irt, 0x1.d0e5600000000p-2 * lt));
    const double k0_f = 0x1.42e730a676c12p+43 * fexp2(fma(-0x1.a0e6900000000p+24, irt, -0x1.347ae20000000p+2 * lt));
    const double kinf_b = 0x1.eddf2cde0c51ep+42 * fexp2(fma(-0x1.06e1a60000000p+27, irt, 0x1.29818a0000000p-4 * lt));
    const double k0_b = 0x1.23bd77a117505p+53 * fexp2(fma(-0x1.1e43fa0000000p+27, irt, -0x1.4ce33e0000000p+2 * lt));
    const double m_ = M9();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.200d1c0000000p-2, fexp2(-(0x1.caf91e3a0f252p-7 * T)), fc);
    fc = fma(0x1.6ff9720000000p-1, fexp2(-(0x1.24f249a032e98p-10 * T)), fc);
    fc = fma(0x1.0000000000000p+0, fexp2(-(0x1.7719c82c0310ap+12 * invT)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C3 * C14 - kb * C17;
    cd3 -= q;
    cd14 -= q;
    cd17 += q;
    }
    {  // R57 (falloff)
    const double kinf_f = 0x1.114edc398b4b1p+33 * fexp2(fma(-0x1.4bf8600000000p+23, irt, 0x1.d0e5600000000p-2 * lt));
    const double k0_f = 0x1.958faf8f67352p+37 * fexp2(fma(-0x1.62f7180000000p+24, irt, -0x1.3333340000000p+2 * lt));
    const double kinf_b = 0x1.8aab8e32c07e1p+46 * fexp2(fma(-0x1.90fa860000000p+26, irt, 0x1.0dbcec0000000p-3 * lt));
    const double k0_b = 0x1.24d431396000fp+51 * fexp2(fma(-0x1.c039400000000p+26, irt, -0x1.47d39a0000000p+2 * lt));
    const double m_ = M10();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.ef9db20000000p-3, fexp2(-(0x1.f6ead796c4570p-7 * T)), fc);
    fc = fma(0x1.8418940000000p-1, fexp2(-(0x1.e66c46e32646ap-11 * T)), fc);
    fc = fma(0x1.0000000000000p+0, fexp2(-(0x1.7ab51b53d1dd2p+12 * invT)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C3 * C14 - kb * C18;
    cd3 -= q;
    cd14 -= q;
    cd18 += q;
    }
    {  // R59 (falloff)
    const double kinf_f = 0x1.63b82ab136e6fp+34 * fexp2(fma(-0x1.5f90000000000p+18, irt, 0x1.0000000000000p-1 * lt));
    const double k0_f = 0x1.40222a3900136p+43 * fexp2(fma(-0x1.4453580000000p+24, irt, -0x1.29999a0000000p+2 * lt));
    const double kinf_b = 0x1.943a01bae3bbep+50 * fexp2(fma(-0x1.8342aa0000000p+28, irt, 0x1.4747b60000000p-1 * lt));
    const double k0_b = 0x1.6bca7591372d2p+59 * fexp2(fma(-0x1.972ffa0000000p+28, irt, -0x1.20b09e0000000p+2 * lt));
    const double m_ = M11();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.99999a0000000p-2, fexp2(-(0x1.d8be0817f5ffep-7 * T)), fc);
    fc = fma(0x1.3333340000000p-1, fexp2(-(0x1.0cf016cf0da73p-16 * T)), fc);
    fc = fma(0x1.0000000000000p+0, fexp2(-(0x1.c2d79a6ff9d67p+13 * invT)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C3 * C17 - kb * C19;
    cd3 -= q;
    cd17 -= q;
    cd19 += q;
    }
    {  // R63 (falloff)
    const double kinf_f = 0x1.c1da4df77dd15p+35 * fexp2(fma(-0x1.9834000000000p+17, irt, 0x1.07ae140000000p-1 * lt));
    const double k0_f = 0x1.7115fca7bac80p+51 * fexp2(fma(-0x1.c1748c0000000p+25, irt, -0x1.dc28f60000000p+2 * lt));
    const double kinf_b = 0x1.3fd7cd950c7b1p+48 * fexp2(fma(-0x1.9e52820000000p+28, irt, 0x1.30b6b60000000p-1 * lt));
    const double k0_b = 0x1.06696cabea55bp+64 * fexp2(fma(-0x1.d64e0c0000000p+28, irt, -0x1.d707f20000000p+2 * lt));
    const double m_ = M12();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.3333340000000p-2, fexp2(-(0x1.d8be0817f5ffep-7 * T)), fc);
    fc = fma(0x1.6666660000000p-1, fexp2(-(0x1.0cf016cf0da73p-16 * T)), fc);
    fc = fma(0x1.0000000000000p+0, fexp2(-(0x1.c2d79a6ff9d67p+13 * invT)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C3 * C18 - kb * C19;
    cd3 -= q;
    cd18 -= q;
    cd19 += q;
    }
    {  // R70 (falloff)
    const double kinf_f = 0x1.6bcc41e900000p+37 * fexp2(fma(0.0, irt, -0x1.0000000000000p+0 * lt));
    const double k0_f = 0x1.518c33f58f036p+48 * fexp2(fma(-0x1.e53ac00000000p+22, irt, -0x1.3333340000000p+2 * lt));
    const double kinf_b = 0x1.97e97ef67bbcdp+54 * fexp2(fma(-0x1.095a0a0000000p+29, irt, -0x1.3f0d840000000p+0 * lt));
    const double k0_b = 0x1.7a7ab5d26528fp+65 * fexp2(fma(-0x1.0d24800000000p+29, irt, -0x1.42f6940000000p+2 * lt));
    const double m_ = M13();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.6a161e0000000p-2, fexp2(-(0x1.66235b77002e7p-7 * T)), fc);
    fc = fma(0x1.4af4f00000000p-1, fexp2(-(0x1.1f99921086155p-10 * T)), fc);
    fc = fma(0x1.0000000000000p+0, fexp2(-(0x1.f5e0a649a80a1p+12 * invT)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C3 * C20 - kb * C21;
    cd3 -= q;
    cd20 -= q;
    cd21 += q;
    }
    {  // R71 (falloff)
    const double kinf_f = 0x1.4dc9380000000p+32 * fexp2(fma(-0x1.3275200000000p+23, irt, 0.0 * lt));
    const double k0_f = 0x1.5baa49ed6ae52p+49 * fexp2(fma(-0x1.ccf0000000000p+24, irt, -0x1.d147ae0000000p+2 * lt));
    const double kinf_b = 0x1.a61a1ee53de0dp+41 * fexp2(fma(-0x1.2b279c0000000p+27, irt, 0x1.6004320000000p-3 * lt));
    const double k0_b = 0x1.b7a505d0e3fbbp+58 * fexp2(fma(-0x1.519e4a0000000p+27, irt, -0x1.c6479a0000000p+2 * lt));
    const double m_ = M14();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.fe91000000000p-3, fexp2(-(0x1.dff101b829d3bp-7 * T)), fc);
    fc = fma(0x1.805bc00000000p-1, fexp2(-(0x1.2278b1ffc7853p-10 * T)), fc);
    fc = fma(0x1.0000000000000p+0, fexp2(-(0x1.77bb5d1fc7413p+12 * invT)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C3 * C21 - kb * C23;
    cd3 -= q;
    cd21 -= q;
    cd23 += q;
    }
    {  // R72 (falloff)
    const double kinf_f = 0x1.e83b7f97942bcp+34 * fexp2(fma(-0x1.1e22000000000p+20, irt, 0x1.147ae20000000p-2 * lt));
    const double k0_f = 0x1.6301b0bd56537p+45 * fexp2(fma(-0x1.a7eb700000000p+23, irt, -0x1.ee147a0000000p+1 * lt));
    const double kinf_b = 0x1.bc2c767d8a9acp+52 * fexp2(fma(-0x1.be06700000000p+28, irt, 0x1.132f020000000p-3 * lt));
    const double k0_b = 0x1.42f9e418789c5p+63 * fexp2(fma(-0x1.ca27aa0000000p+28, irt, -0x1.ff70ce0000000p+1 * lt));
    const double m_ = M15();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.be76c80000000p-3, fexp2(-(0x1.c7a7bdc6e6f07p-8 * T)), fc);
    fc = fma(0x1.90624e0000000p-1, fexp2(-(0x1.1c09331a387a3p-11 * T)), fc);
    fc = fma(0x1.0000000000000p+0, fexp2(-(0x1.12c9cf68db79ep+13 * invT)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C3 * C23 - kb * C25;
    cd3 -= q;
    cd23 -= q;
    cd25 += q;
    }
    {  // R74 (falloff)
    const double kinf_f = 0x1.114edc398b4b1p+33 * fexp2(fma(-0x1.d0c8600000000p+22, irt, 0x1.d0e5600000000p-2 * lt));
    const double k0_f = 0x1.3535f6503834dp+50 * fexp2(fma(-0x1.bcfa100000000p+24, irt, -0x1.e7ae140000000p+2 * lt));
    const double kinf_b = 0x1.d3efa52e47385p+42 * fexp2(fma(-0x1.2f2d980000000p+27, irt, 0x1.54abe60000000p-2 * lt));
    const double k0_b = 0x1.08b520c224c76p+60 * fexp2(fma(-0x1.5846960000000p+27, irt, -0x1.ef71a00000000p+2 * lt));
    const double m_ = M16();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.94af500000000p-6, fexp2(-(0x1.c23b13e60edb5p-8 * T)), fc);
    fc = fma(0x1.f35a860000000p-1, fexp2(-(0x1.8057e54783511p-10 * T)), fc);
    fc = fma(0x1.0000000000000p+0, fexp2(-(0x1.8a6591da95702p+12 * invT)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C3 * C25 - kb * C26;
    cd3 -= q;
    cd25 -= q;
    cd26 += q;
    }
    {  // R76 (falloff)
    const double kinf_f = 0x1.f8592ae3e59d9p+39 * fexp2(fma(-0x1.9380e00000000p+22, irt, -0x1.fae1480000000p-1 * lt));
    const double k0_f = 0x1.744837ad03a96p+53 * fexp2(fma(-0x1.aac9d00000000p+24, irt, -0x1.c51eb80000000p+2 * lt));
    const double kinf_b = 0x1.449a77c0f0282p+58 * fexp2(fma(-0x1.9871fe0000000p+28, irt, -0x1.32edbc0000000p+0 * lt));
    const double k0_b = 0x1.df3568c455bf9p+71 * fexp2(fma(-0x1.acd0980000000p+28, irt, -0x1.d27dfe0000000p+2 * lt));
    const double m_ = M17();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.432ca60000000p-3, fexp2(-(0x1.7a31a0132b331p-7 * T)), fc);
    fc = fma(0x1.af34d60000000p-1, fexp2(-(0x1.54de64aaf2369p-11 * T)), fc);
    fc = fma(0x1.0000000000000p+0, fexp2(-(0x1.364504a6dddbcp+13 * invT)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C3 * C26 - kb * C27;
    cd3 -= q;
    cd26 -= q;
    cd27 += q;
    }
    {  // R83 (falloff)
    const double kinf_f = 0x1.db165dca09689p+28 * fexp2(fma(-0x1.3d9e0f0000000p+28, irt, 0x1.8000000000000p+0 * lt));
    const double k0_f = 0x1.401f1048f94bbp+41 * fexp2(fma(-0x1.50921c0000000p+28, irt, -0x1.b5c2900000000p+1 * lt));
    const double kinf_b = 0x1.470b40dce8b8fp+44 * fexp2(fma(-0x1.3fcc880000000p+28, irt, 0x1.a2bb440000000p-1 * lt));
    const double k0_b = 0x1.b8b8a66e1e59fp+56 * fexp2(fma(-0x1.52c0940000000p+28, irt, -0x1.0689f40000000p+2 * lt));
    const double m_ = M18();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.16872c0000000p-4, fexp2(-(0x1.dff101b829d3bp-8 * T)), fc);
    fc = fma(0x1.dd2f1a0000000p-1, fexp2(-(0x1.eb292cfaf8ef3p-11 * T)), fc);
    fc = fma(0x1.0000000000000p+0, fexp2(-(0x1.d05e124541553p+13 * invT)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C5 * C9 - kb * C14;
    cd5 -= q;
    cd9 -= q;
    cd14 += q;
    }
    {  // R85 (falloff)
    const double kinf_f = 0x1.b69d09bfd6015p+32 * fexp2(fma(0.0, irt, -0x1.7ae1480000000p-2 * lt));
    const double k0_f = 0x1.f3a6262a20a58p+32 * fexp2(fma(0x1.b224a00000000p+22, irt, -0x1.cccccc0000000p-1 * lt));
    const double kinf_b = 0x1.02e707efb45d3p+52 * fexp2(fma(-0x1.a070e40000000p+27, irt, -0x1.63f9c60000000p+0 * lt));
    const double k0_b = 0x1.26ee24007b566p+52 * fexp2(fma(-0x1.92dfbe0000000p+27, irt, -0x1.eba7da0000000p+0 * lt));
    const double m_ = M19();
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
    const double q = kf * C4 * C4 - kb * C7;
    cd4 = fma(-0x1.0000000000000p+1, q, cd4);
    cd7 += q;
    }
    {  // R95 (falloff)
    const double kinf_f = 0x1.5b1855c77e0ddp+38 * fexp2(fma(-0x1.53a9200000000p+22, irt, -0x1.6e147a0000000p+0 * lt));
    const double k0_f = 0x1.4ca546554ff35p+48 * fexp2(fma(-0x1.90f0a00000000p+23, irt, -0x1.7ae1480000000p+2 * lt));
    const double kinf_b = 0x1.11126ffeb5740p+59 * fexp2(fma(-0x1.7b4c5c0000000p+28, irt, -0x1.21ac9a0000000p+1 * lt));
    const double k0_b = 0x1.05b44e174f6d3p+69 * fexp2(fma(-0x1.82853c0000000p+28, irt, -0x1.b032760000000p+2 * lt));
    const double m_ = M20();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.2d0e560000000p-1, fexp2(-(0x1.e4dd291f23b11p-8 * T)), fc);
    fc = fma(0x1.a5e3540000000p-2, fexp2(-(0x1.006711681d49bp-12 * T)), fc);
    fc = fma(0x1.0000000000000p+0, fexp2(-(0x1.2044bc9a7062ep+13 * invT)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C4 * C13 - kb * C19;
    cd4 -= q;
    cd13 -= q;
    cd19 += q;
    }
    {  // R131 (falloff)
    const double kinf_f = 0x1.74876e8000000p+35 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double k0_f = 0x1.cd72ae192db6ap+40 * fexp2(fma(-0x1.ee62800000000p+22, irt, -0x1.deb8520000000p+1 * lt));
    const double kinf_b = 0x1.8fb4cbb0d0cd3p+54 * fexp2(fma(-0x1.2a30e00000000p+28, irt, -0x1.70e3680000000p+0 * lt));
    const double k0_b = 0x1.ef1c822e7b8bap+59 * fexp2(fma(-0x1.31ea6a0000000p+28, irt, -0x1.4b95040000000p+2 * lt));
    const double m_ = M21();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.b27bb20000000p-2, fexp2(-(0x1.8ef04bf5f9b89p-8 * T)), fc);
    fc = fma(0x1.26c2260000000p-1, fexp2(-(0x1.c9dc9f1558df0p-11 * T)), fc);
    fc = fma(0x1.0000000000000p+0, fexp2(-(0x1.c91056ae3e90cp+12 * invT)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C8 * C9 - kb * C22;
    cd8 -= q;
    cd9 -= q;
    cd22 += q;
    }
    {  // R140 (falloff)
    const double kinf_f = 0x1.111c906616bd7p+34 * fexp2(fma(-0x1.1feef00000000p+24, irt, 0x1.0000000000000p-1 * lt));
    const double k0_f = 0x1.1812e88a3b07ep+45 * fexp2(fma(-0x1.c4f5080000000p+24, irt, -0x1.470a3e0000000p+2 * lt));
    const double kinf_b = 0x1.b6aea43f0f007p+56 * fexp2(fma(-0x1.5171860000000p+28, irt, -0x1.3ee43a0000000p+0 * lt));
    const double k0_b = 0x1.c1dd98ab88dd9p+67 * fexp2(fma(-0x1.5bc1e60000000p+28, irt, -0x1.b6c34c0000000p+2 * lt));
    const double m_ = M22();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.a31f8a0000000p-2, fexp2(-(0x1.57d005e2e1744p-8 * T)), fc);
    fc = fma(0x1.2e703a0000000p-1, fexp2(-(0x1.347a54a0f762ep-10 * T)), fc);
    fc = fma(0x1.0000000000000p+0, fexp2(-(0x1.d385fb0816482p+12 * invT)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C10 * C9 - kb * C24;
    cd9 -= q;
    cd10 -= q;
    cd24 += q;
    }
    {  // R147 (falloff)
    const double kinf_f = 0x1.43247c05cf3f1p+38 * fexp2(fma(-0x1.246b600000000p+22, irt, -0x1.28f5c20000000p+0 * lt));
    const double k0_f = 0x1.f64f07f87c742p+49 * fexp2(fma(-0x1.41c3180000000p+24, irt, -0x1.970a3e0000000p+2 * lt));
    const double kinf_b = 0x1.795a74a0bde05p+59 * fexp2(fma(-0x1.7ddc420000000p+28, irt, -0x1.3c255c0000000p+1 * lt));
    const double k0_b = 0x1.2549fc4a02a30p+71 * fexp2(fma(-0x1.8d66c60000000p+28, irt, -0x1.eadf7a0000000p+2 * lt));
    const double m_ = M23();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.96d5d00000000p-2, fexp2(-(0x1.c68f568d31760p-8 * T)), fc);
    fc = fma(0x1.3495180000000p-1, fexp2(-(0x1.81b71db5d175cp-12 * T)), fc);
    fc = fma(0x1.0000000000000p+0, fexp2(-(0x1.caf515898b228p+13 * invT)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C12 * C28 - kb * C19;
    cd12 -= q;
    cd19 += q;
    cd28 -= q;
    }
    {  // R158 (falloff)
    const double kinf_f = 0x1.408254d335683p+35 * fexp2(fma(-0x1.4dfc000000000p+21, irt, -0x1.2e147a0000000p+0 * lt));
    const double k0_f = 0x1.b270dffb6e516p+54 * fexp2(fma(-0x1.60a9400000000p+23, irt, -0x1.c1eb860000000p+2 * lt));
    const double kinf_b = 0x1.4020441da519fp+60 * fexp2(fma(-0x1.719e724000000p+28, irt, -0x1.4860020000000p+1 * lt));
    const double k0_b = 0x1.b1ec086a95561p+79 * fexp2(fma(-0x1.7a07c44000000p+28, irt, -0x1.0d4b340000000p+3 * lt));
    const double m_ = M24();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.8624de0000000p-2, fexp2(-(0x1.42e95359bf579p-6 * T)), fc);
    fc = fma(0x1.3ced920000000p-1, fexp2(-(0x1.4080d5c2249c2p-10 * T)), fc);
    fc = fma(0x1.0000000000000p+0, fexp2(-(0x1.c2cc0fcc4740bp+13 * invT)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C13 * C13 - kb * C27;
    cd13 = fma(-0x1.0000000000000p+1, q, cd13);
    cd27 += q;
    }
    {  // R167 (third_body)
    const double kf = 0x1.5426a92560000p+38 * fexp2(fma(-0x1.0f54f00000000p+26, irt, -0x1.0000000000000p+0 * lt));
    const double kb = 0x1.18d7f8975dd24p+28 * fexp2(fma(-0x1.46cef00000000p+22, irt, -0x1.88d9fa0000000p-1 * lt));
    const double q = (kf * C11 - kb * C9 * C3) * M25();
    cd3 += q;
    cd9 += q;
    cd11 -= q;
    }
    {  // R174 (falloff)
    const double kinf_f = 0x1.c4ed80e7a3586p+46 * fexp2(fma(-0x1.5a3a470000000p+28, irt, 0x1.c28f5c0000000p-2 * lt));
    const double k0_f = 0x1.54ba0c24c71b7p+76 * fexp2(fma(-0x1.863d1f8000000p+28, irt, -0x1.29999a0000000p+3 * lt));
    const double kinf_b = 0x1.8f6a2d9e2ba19p+30 * fexp2(fma(-0x1.5cb21c0000000p+27, irt, 0x1.820a520000000p-1 * lt));
    const double k0_b = 0x1.2c7b0f65c35bbp+60 * fexp2(fma(-0x1.b4b7ce0000000p+27, irt, -0x1.1f8d640000000p+3 * lt));
    const double m_ = M26();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.0fdf3c0000000p-2, fexp2(-(0x1.06a2764633554p-7 * T)), fc);
    fc = fma(0x1.7810620000000p-1, fexp2(-(0x1.6d67996cccfc3p-10 * T)), fc);
    fc = fma(0x1.0000000000000p+0, fexp2(-(0x1.e87143bbc5b6dp+12 * invT)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C25 - kb * C21 * C5;
    cd5 += q;
    cd21 += q;
    cd25 -= q;
    }
    {  // R289 (falloff)
    const double kinf_f = 0x1.ad366b951da24p+34 * fexp2(fma(0x1.79ee000000000p+20, irt, 0x1.b851ec0000000p-2 * lt));
    const double k0_f = 0x1.2328e8c9877bap+40 * fexp2(fma(-0x1.2d64400000000p+21, irt, -0x1.6666660000000p+1 * lt));
    const double kinf_b = 0x1.3552dfff27e7cp+51 * fexp2(fma(-0x1.ae52540000000p+28, irt, -0x1.02cc980000000p-5 * lt));
    const double k0_b = 0x1.a3ab36e8f59b4p+56 * fexp2(fma(-0x1.b2270a0000000p+28, irt, -0x1.a17bc80000000p+1 * lt));
    const double m_ = M27();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.b020c40000000p-2, fexp2(-(0x1.837e62f643580p-7 * T)), fc);
    fc = fma(0x1.27ef9e0000000p-1, fexp2(-(0x1.2a60b6d815f6dp-11 * T)), fc);
    fc = fma(0x1.0000000000000p+0, fexp2(-(0x1.a636b664005f8p+13 * invT)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C8 * C5 - kb * C13;
    cd5 -= q;
    cd8 -= q;
    cd13 += q;
    }
    {  // R304 (falloff)
    const double kinf_f = 0x1.9357e28947c6ep+32 * fexp2(fma(0x1.c02e600000000p+22, irt, 0x1.b020c40000000p-2 * lt));
    const double k0_f = 0x1.e9fe697d920c9p+50 * fexp2(fma(-0x1.ec18900000000p+23, irt, -0x1.e851ec0000000p+2 * lt));
    const double kinf_b = 0x1.018dea56ff687p+43 * fexp2(fma(-0x1.06e3ba0000000p+27, irt, 0x1.d8e9f60000000p-2 * lt));
    const double k0_b = 0x1.38e2a4fa5d55bp+61 * fexp2(fma(-0x1.33a6b60000000p+27, irt, -0x1.e5c5580000000p+2 * lt));
    const double m_ = M28();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.11eb860000000p-1, fexp2(-(0x1.d663ee94a85b9p-8 * T)), fc);
    fc = fma(0x1.dc28f60000000p-2, fexp2(-(0x1.aa9d56dc96f51p-11 * T)), fc);
    fc = fma(0x1.0000000000000p+0, fexp2(-(0x1.e0de484e936fdp+12 * invT)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C3 * C24 - kb * C32;
    cd3 -= q;
    cd24 -= q;
    cd32 += q;
    }
    {  // R312 (falloff)
    const double kinf_f = 0x1.190930c000000p+33 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double k0_f = 0x1.ee5b180027f0fp+75 * fexp2(fma(-0x1.a10da00000000p+25, irt, -0x1.0d1eb80000000p+4 * lt));
    const double kinf_b = 0x1.a58242336af06p+59 * fexp2(fma(-0x1.6635f40000000p+28, irt, -0x1.c2e1f00000000p+0 * lt));
    const double k0_b = 0x1.72a1e7f557044p+102 * fexp2(fma(-0x1.9a57a80000000p+28, irt, -0x1.294d020000000p+4 * lt));
    const double m_ = M29();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.b1d14e0000000p-1, fexp2(-(0x1.44e8a76e993cap-8 * T)), fc);
    fc = fma(0x1.38bac80000000p-3, fexp2(-(0x1.13da40d9236e4p-11 * T)), fc);
    fc = fma(0x1.0000000000000p+0, fexp2(-(0x1.5d500268fc745p+13 * invT)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C13 * C26 - kb * C34;
    cd13 -= q;
    cd26 -= q;
    cd34 += q;
    }
    {  // R318 (falloff)
    const double kinf_f = 0x1.a497dc8d74d43p+25 * fexp2(fma(-0x1.6be8280000000p+24, irt, 0x1.99999a0000000p+0 * lt));
    const double k0_f = 0x1.72e4b0a726b5dp+59 * fexp2(fma(-0x1.2201360000000p+26, irt, -0x1.d333340000000p+3 * lt));
    const double kinf_b = 0x1.5d6e5f2c5857ep+43 * fexp2(fma(-0x1.e537540000000p+26, irt, -0x1.ea0f320000000p-5 * lt));
    const double k0_b = 0x1.342eca62b2986p+77 * fexp2(fma(-0x1.561f400000000p+27, irt, -0x1.0428240000000p+4 * lt));
    const double m_ = M30();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.9f06f60000000p-1, fexp2(-(0x1.5554873ae385ep-8 * T)), fc);
    fc = fma(0x1.83e4260000000p-3, fexp2(-(0x1.59db35901107fp-13 * T)), fc);
    fc = fma(0x1.0000000000000p+0, fexp2(-(0x1.63c273d9be1b6p+13 * invT)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C13 * C25 - kb * C35;
    cd13 -= q;
    cd25 -= q;
    cd35 += q;
    }
    {  // R320 (falloff)
    const double kinf_f = 0x1.0d30819000000p+35 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double k0_f = 0x1.ece120f942710p+62 * fexp2(fma(-0x1.6a88980000000p+25, irt, -0x1.b170a40000000p+3 * lt));
    const double kinf_b = 0x1.a003bd965091cp+53 * fexp2(fma(-0x1.93fa4c2000000p+28, irt, -0x1.c831ae0000000p-3 * lt));
    const double k0_b = 0x1.7cbd45b8f67c5p+81 * fexp2(fma(-0x1.c14b5f2000000p+28, irt, -0x1.b891d20000000p+3 * lt));
    const double m_ = M31();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.5eb8520000000p-1, fexp2(-(0x1.003a98da578b6p-8 * T)), fc);
    fc = fma(0x1.428f5c0000000p-2, fexp2(-(0x1.cc829042fb52ep-12 * T)), fc);
    fc = fma(0x1.0000000000000p+0, fexp2(-(0x1.2c93952be2163p+13 * invT)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C3 * C35 - kb * C34;
    cd3 -= q;
    cd34 += q;
    cd35 -= q;
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
    cd[9] = cd9;
    cd[10] = cd10;
    cd[11] = cd11;
    cd[12] = cd12;
    cd[13] = cd13;
    cd[14] = cd14;
    cd[15] = cd15;
    cd[16] = cd16;
    cd[17] = cd17;
    cd[18] = cd18;
    cd[19] = cd19;
    cd[20] = cd20;
    cd[21] = cd21;
    cd[22] = cd22;
    cd[23] = cd23;
    cd[24] = cd24;
    cd[25] = cd25;
    cd[26] = cd26;
    cd[27] = cd27;
    cd[28] = cd28;
    cd[29] = cd29;
    cd[30] = cd30;
    cd[31] = cd31;
    cd[32] = cd32;
    cd[33] = cd33;
    cd[34] = cd34;
    cd[35] = cd35;
  }

  // s: [rho*Y (36), rho*T] of this lane's state; f: the right-hand side
  static __device__ __forceinline__ void eval(const double (&s)[37], double P, double (&f)[37]) {
    double rho = s[0];
    rho += s[1];
    rho += s[2];
    rho += s[3];
    rho += s[4];
    rho += s[5];
    rho += s[6];
    rho += s[7];
    rho += s[8];
    rho += s[9];
    rho += s[10];
    rho += s[11];
    rho += s[12];
    rho += s[13];
    rho += s[14];
    rho += s[15];
    rho += s[16];
    rho += s[17];
    rho += s[18];
    rho += s[19];
    rho += s[20];
    rho += s[21];
    rho += s[22];
    rho += s[23];
    rho += s[24];
    rho += s[25];
    rho += s[26];
    rho += s[27];
    rho += s[28];
    rho += s[29];
    rho += s[30];
    rho += s[31];
    rho += s[32];
    rho += s[33];
    rho += s[34];
    rho += s[35];
    const double T = s[36] / rho;
    const double irho = 1.0 / rho;
    double C[36], cd[36];
    C[0] = s[0] * 0x1.245cd2eb40a46p-5;
    C[1] = s[1] * 0x1.0000000000000p-4;
    C[2] = s[2] * 0x1.0000000000000p-5;
    C[3] = s[3] * 0x1.fbefbe72dfd0bp-1;
    C[4] = s[4] * 0x1.e1a7dc7865ca7p-5;
    C[5] = s[5] * 0x1.fbefbe72dfd0bp-2;
    C[6] = s[6] * 0x1.f05d519a5a4afp-6;
    C[7] = s[7] * 0x1.e1a7dc7865ca7p-6;
    C[8] = s[8] * 0x1.3aa42a8f7dbc3p-4;
    C[9] = s[9] * 0x1.24778b96770f5p-5;
    C[10] = s[10] * 0x1.24077255ac595p-4;
    C[11] = s[11] * 0x1.1a4ebab921f45p-5;
    C[12] = s[12] * 0x1.24077255ac595p-4;
    C[13] = s[13] * 0x1.1072f8c06c358p-4;
    C[14] = s[14] * 0x1.10d4897263b9dp-5;
    C[15] = s[15] * 0x1.fea8d69a8976dp-5;
    C[16] = s[16] * 0x1.74476f46bcafbp-6;
    C[17] = s[17] * 0x1.07f7f2b66042cp-5;
    C[18] = s[18] * 0x1.07f7f2b66042cp-5;
    C[19] = s[19] * 0x1.ff5431b9fabeep-6;
    C[20] = s[20] * 0x1.47503bacf8495p-5;
    C[21] = s[21] * 0x1.3aa42a8f7dbc3p-5;
    C[22] = s[22] * 0x1.8f56483547455p-6;
    C[23] = s[23] * 0x1.2ee9ec61a82a7p-5;
    C[24] = s[24] * 0x1.85c2db9e52812p-6;
    C[25] = s[25] * 0x1.24077255ac595p-5;
    C[26] = s[26] * 0x1.19e6472ab1c54p-5;
    C[27] = s[27] * 0x1.1072f8c06c358p-5;
    C[28] = s[28] * 0x1.c6b4f7f1539dfp-5;
    C[29] = s[29] * 0x1.9a221661a2c13p-6;
    C[30] = s[30] * 0x1.550c9313ea131p-4;
    C[31] = s[31] * 0x1.85c2db9e52812p-6;
    C[32] = s[32] * 0x1.7ca23f7ff2a8bp-6;
    C[33] = s[33] * 0x1.73ec922c64208p-6;
    C[34] = s[34] * 0x1.7391df46c8924p-6;
    C[35] = s[35] * 0x1.7c434324c92a8p-6;
    const bool hi = T > 0x1.f400000000000p+9;
    double cpm = 0.0;
    if (hi) {
      cpm = fma(s[0] * irho, 0x1.28ba9057d1783p+8 * (0x1.769c23b7952d2p+1 + T * (0x1.86106ec5d7fc6p-10 + T * (-0x1.3132bf1b89c39p-21 + T * (0x1.bc128a9b8a724p-34 + T * -0x1.e6a15668d1fd9p-48)))), cpm);
      cpm = fma(s[1] * irho, 0x1.03d2b851eb852p+9 * (0x1.48e2c7b5e1a3dp+1 + T * (-0x1.689a006cdb509p-14 + T * (0x1.6855a2fbdda5cp-25 + T * (-0x1.607823c010ceap-37 + T * 0x1.620b4436bd152p-50)))), cpm);
      cpm = fma(s[2] * irho, 0x1.03d2b851eb852p+8 * (0x1.a42a332f575b8p+1 + T * (0x1.84c851ecf574dp-10 + T * (-0x1.96ee255022a3dp-21 + T * (0x1.cca1706e20348p-33 + T * -0x1.8667712a69c18p-46)))), cpm);
      cpm = fma(s[3] * irho, 0x1.01c2d34acaff7p+13 * (0x1.40000015798eep+1 + T * (-0x1.961a6ec6a1e45p-36 + T * (0x1.230b4c341c642p-46 + T * (-0x1.5d647fbe2e672p-58 + T * 0x1.2d244e9510ba2p-71)))), cpm);
      cpm = fma(s[4] * irho, 0x1.e8d949731098dp+8 * (0x1.8be3be406d029p+1 + T * (0x1.1f88fd8e1440ep-11 + T * (0x1.0faafc0d73234p-23 + T * (-0x1.82ca91827ab6dp-34 + T * 0x1.a705cd746f5f8p-47)))), cpm);
      cpm = fma(s[5] * irho, 0x1.01c2d350092cdp+12 * (0x1.ab2bf6fecf7e5p+1 + T * (-0x1.9e6b00cea2ba4p-15 + T * (0x1.0c24d11e93b22p-21 + T * (-0x1.8adee4a4b6baep-33 + T * 0x1.68bf7de4136dcp-46)))), cpm);
      cpm = fma(s[6] * irho, 0x1.f7c6fae7924afp+7 * (0x1.0119fbbf289f6p+2 + T * (0x1.2593e46a1f9dfp-9 + T * (-0x1.5431502070c84p-21 + T * (0x1.f675fa32f618cp-34 + T * -0x1.84c80e71ea191p-47)))), cpm);
      cpm = fma(s[7] * irho, 0x1.e8d94983d7907p+7 * (0x1.0a8f681d1fcb7p+2 + T * (0x1.41abe4bc5704bp-8 + T * (-0x1.fe66ae3495cc5p-20 + T * (0x1.981f91177d524p-32 + T * -0x1.0353229ef325dp-45)))), cpm);
      cpm = fma(s[8] * irho, 0x1.3f5713b5bf6a1p+9 * (0x1.70718843050d6p+1 + T * (0x1.fd09d40e9c422p-11 + T * (0x1.3631d6b0442c1p-23 + T * (-0x1.1f62b7f017dbdp-33 + T * 0x1.3d32486a4348dp-46)))), cpm);
      cpm = fma(s[9] * irho, 0x1.28d5af07bfe7ep+8 * (0x1.5b8b33bac2892p+1 + T * (0x1.0e56efb7c8adbp-9 + T * (-0x1.0c1ec8ca156a0p-20 + T * (0x1.f9e45483ed15bp-33 + T * -0x1.6edbeeb572dccp-46)))), cpm);
      cpm = fma(s[10] * irho, 0x1.2863e90ff9724p+9 * (0x1.6fe28bbb5f921p+1 + T * (0x1.df4030068403dp-9 + T * (-0x1.7a3607a17a275p-20 + T * (0x1.1e1208519dbd9p-32 + T * -0x1.522e0f41fe4e3p-46)))), cpm);
      cpm = fma(s[11] * irho, 0x1.1e860685553efp+8 * (0x1.62d69c2e745cap+1 + T * (0x1.44dbe8babc438p-8 + T * (-0x1.4d75433aa4a6fp-19 + T * (0x1.43e5261c638b2p-31 + T * -0x1.e08abbb0771a1p-45)))), cpm);
      cpm = fma(s[12] * irho, 0x1.2863e90ff9724p+9 * (0x1.256183d389aa6p+1 + T * (0x1.3120cfb16b35fp-8 + T * (-0x1.0e0906cfb21aep-19 + T * (0x1.cb7e14e4de1f4p-32 + T * -0x1.31fd42b26d354p-45)))), cpm);
      cpm = fma(s[13] * irho, 0x1.148494a2b9d3dp+9 * (0x1.249265f3a4d2ep+1 + T * (0x1.da795f50c1384p-8 + T * (-0x1.90ed77ebb7110p-19 + T * (0x1.477b292040de5p-31 + T * -0x1.a4c6782829ae7p-45)))), cpm);
      cpm = fma(s[14] * irho, 0x1.14e7994e1a3f4p+8 * (0x1.c2bc95c7fddb1p+0 + T * (0x1.2d77335291c21p-7 + T * (-0x1.28cb7c4b91fedp-18 + T * (0x1.14a3f4fe94722p-30 + T * -0x1.8e0d9e100cd20p-44)))), cpm);
      cpm = fma(s[15] * irho, 0x1.03249374bc6a8p+9 * (0x1.32977b314eac9p-4 + T * (0x1.b6cb6711ca116p-7 + T * (-0x1.80b9c08579157p-18 + T * (0x1.5027b89a2ce85p-30 + T * -0x1.ca88f7d990082p-44)))), cpm);
      cpm = fma(s[16] * irho, 0x1.79d6b356da017p+7 * (0x1.edc1423f95973p+1 + T * (0x1.214cd7e62db66p-8 + T * (-0x1.29446e529e95bp-19 + T * (0x1.1fcab1b9912a3p-31 + T * -0x1.a937326a2284cp-45)))), cpm);
      cpm = fma(s[17] * irho, 0x1.0be922424a277p+8 * (0x1.d8a944f2ce3e4p+1 + T * (0x1.1b4df55708be3p-7 + T * (-0x1.f773c3714a914p-19 + T * (0x1.b0c96ce8203e2p-31 + T * -0x1.24153561cd7f6p-44)))), cpm);
      cpm = fma(s[18] * irho, 0x1.0be922424a277p+8 * (0x1.e2a98aa8650e7p+1 + T * (0x1.01eee717c07fdp-7 + T * (-0x1.6488a8c446c70p-19 + T * (0x1.b1b1dcc557332p-32 + T * -0x1.7c93377953d3bp-46)))), cpm);
      cpm = fma(s[19] * irho, 0x1.037b88a8b08ddp+8 * (0x1.ca2a4c2ed7aedp+0 + T * (0x1.cdd39bbea4fb5p-7 + T * (-0x1.ab2602c451494p-18 + T * (0x1.7bcd41e074550p-30 + T * -0x1.07989f5b3e268p-43)))), cpm);
      cpm = fma(s[20] * irho, 0x1.4c3397bb73083p+8 * (0x1.957aaf1dba502p+1 + T * (0x1.377101463a6fcp-8 + T * (-0x1.ed598482ed583p-20 + T * (0x1.4e75f1b05c789p-32 + T * -0x1.3f4630515edadp-46)))), cpm);
      cpm = fma(s[21] * irho, 0x1.3f5713ad5bee4p+8 * (0x1.0971c7ee6bae0p+2 + T * (0x1.86b42b3f9ab1ep-8 + T * (-0x1.3e7de3eb387edp-19 + T * (0x1.00f66a3bafde2p-31 + T * -0x1.455f2b475f023p-45)))), cpm);
      cpm = fma(s[22] * irho, 0x1.954cff43419e3p+7 * (0x1.683486198a14cp+2 + T * (0x1.0bbca21f5e9bfp-8 + T * (-0x1.abbd5f8926da2p-20 + T * (0x1.3abf2c56d8d5fp-32 + T * -0x1.5d9ed3d5e2c0fp-46)))), cpm);
      cpm = fma(s[23] * irho, 0x1.33700096feb4ap+8 * (0x1.8224031487768p+1 + T * (0x1.52803e497ede9p-7 + T * (-0x1.3a1fef6b5677dp-18 + T * (0x1.17b98c3c9686ep-30 + T * -0x1.847bd21d4a0a4p-44)))), cpm);
      cpm = fma(s[24] * irho, 0x1.8b94f63800219p+7 * (0x1.20b91864fbad3p+2 + T * (0x1.2707a64c0b6f9p-7 + T * (-0x1.17cdaf120e12fp-18 + T * (0x1.fb9d615c62415p-31 + T * -0x1.65f69aff87e86p-44)))), cpm);
      cpm = fma(s[25] * irho, 0x1.2863e90ff9724p+8 * (0x1.049f4a5d9c3d6p+1 + T * (0x1.dfe6a5720731ep-7 + T * (-0x1.c25a4ed3d3908p-18 + T * (0x1.94aeec0be93f2p-30 + T * -0x1.1b109c49479cdp-43)))), cpm);
      cpm = fma(s[26] * irho, 0x1.1e1c0389f83bep+8 * (0x1.f4645cf6d1024p+0 + T * (0x1.1d0972c8defc6p-6 + T * (-0x1.0bd56e41b638fp-17 + T * (0x1.e1a27cc16cb18p-30 + T * -0x1.50f67ed791cc7p-43)))), cpm);
      cpm = fma(s[27] * irho, 0x1.148494a2b9d3dp+8 * (0x1.1266d373affb0p+0 + T * (0x1.634a9ae4e575dp-6 + T * (-0x1.50674e48c90f9p-17 + T * (0x1.304e6c1a9e602p-29 + T * -0x1.abd9357b132f9p-43)))), cpm);
      cpm = fma(s[28] * irho, 0x1.cd7f5ff609dd0p+8 * (0x1.8459ddac6e07ap+1 + T * (0x1.1d553f9364039p-9 + T * (-0x1.6057d217698d4p-23 + T * (-0x1.aacb906a5f7ccp-34 + T * 0x1.2f01042cd6ffep-46)))), cpm);
      cpm = fma(s[29] * irho, 0x1.a04215336deb9p+7 * (0x1.4000000000000p+1 + T * (0.0 + T * (0.0 + T * (0.0 + T * 0.0)))), cpm);
      cpm = fma(s[30] * irho, 0x1.5a24731d2e0e3p+9 * (0x1.3f0fc61badb08p+1 + T * (0x1.928f7063e1320p-15 + T * (-0x1.37197a49dc877p-24 + T * (0x1.493ad8d0d6b66p-35 + T * -0x1.5f1ee7e5c04b1p-48)))), cpm);
      cpm = fma(s[31] * irho, 0x1.8b94f63800219p+7 * (0x1.7b200416e5f59p+2 + T * (0x1.bd24e4100a643p-8 + T * (-0x1.58622793768ddp-19 + T * (0x1.eea583d58eb03p-32 + T * -0x1.0dad2c2e98a20p-45)))), cpm);
      cpm = fma(s[32] * irho, 0x1.825174a3400b9p+7 * (0x1.7e7160956c0d7p+2 + T * (0x1.0a6c5738986f4p-7 + T * (-0x1.703e33ec05ba6p-19 + T * (0x1.bf88df5305066p-32 + T * -0x1.87ff125e0d08ep-46)))), cpm);
      cpm = fma(s[33] * irho, 0x1.797a7aa68f4b6p+7 * (0x1.59dcf38b7d772p+2 + T * (0x1.80242581cd52bp-7 + T * (-0x1.1b9f84391e21fp-18 + T * (0x1.77e1ab96723c6p-31 + T * -0x1.7128a8eac22f7p-45)))), cpm);
      cpm = fma(s[34] * irho, 0x1.791e6f0cfe154p+7 * (0x1.e22f4c1de5c41p+2 + T * (0x1.3533e853aabbcp-6 + T * (-0x1.a4e58c0d6bc65p-18 + T * (0x1.f6e487e665bdbp-31 + T * -0x1.aee313b4d365ep-45)))), cpm);
      cpm = fma(s[35] * irho, 0x1.81f10d173fb7ap+7 * (0x1.ecf903f7dc451p+2 + T * (0x1.06de43cb39826p-6 + T * (-0x1.628ec7e39e9d3p-18 + T * (0x1.a374b81e9310cp-31 + T * -0x1.62d06c34a626ep-45)))), cpm);
    } else {
      cpm = fma(s[0] * irho, 0x1.28ba9057d1783p+8 * (0x1.a63b0c4588a05p+1 + T * (0x1.712969da04050p-10 + T * (-0x1.09f7a2b098bd4p-18 + T * (0x1.83ae94da0fe59p-28 + T * -0x1.581526048e0d6p-39)))), cpm);
      cpm = fma(s[1] * irho, 0x1.03d2b851eb852p+9 * (0x1.9589c6bdbf12dp+1 + T * (-0x1.add3ae5787a18p-9 + T * (0x1.bdcef845b6ae0p-18 + T * (-0x1.a51e14d5c0503p-28 + T * 0x1.2954967e1b470p-39)))), cpm);
      cpm = fma(s[2] * irho, 0x1.03d2b851eb852p+8 * (0x1.e42787ae5fa45p+1 + T * (-0x1.88c9b66c8c0dfp-9 + T * (0x1.4a6bae1fdae75p-17 + T * (-0x1.4ca5927ada53cp-27 + T * 0x1.c883a18b02bcdp-39)))), cpm);
      cpm = fma(s[3] * irho, 0x1.01c2d34acaff7p+13 * (0x1.4000000000000p+1 + T * (0x1.8d112bff6d580p-41 + T * (-0x1.1fa470055807fp-49 + T * (0x1.538a620b2373fp-59 + T * -0x1.1863cffe0b329p-70)))), cpm);
      cpm = fma(s[4] * irho, 0x1.e8d949731098dp+8 * (0x1.fefa5c927d1abp+1 + T * (-0x1.3abed86e71c7dp-9 + T * (0x1.35e793e99fbcdp-18 + T * (-0x1.0ab59e9e67441p-28 + T * 0x1.7ff6d2c211dd3p-40)))), cpm);
      cpm = fma(s[5] * irho, 0x1.01c2d350092cdp+12 * (0x1.2c130ac9b2911p+1 + T * (0x1.058175d02a941p-7 + T * (-0x1.46ca05831775cp-16 + T * (0x1.5a4c582f87e3dp-26 + T * -0x1.03862939e564dp-37)))), cpm);
      cpm = fma(s[6] * irho, 0x1.f7c6fae7924afp+7 * (0x1.1350a899bcaa1p+2 + T * (-0x1.373d054674594p-8 + T * (0x1.62fa28e3a8ea6p-16 + T * (-0x1.a110b0905e0fcp-26 + T * 0x1.46f1288fc5c1cp-37)))), cpm);
      cpm = fma(s[7] * irho, 0x1.e8d94983d7907p+7 * (0x1.11abd48f63e0ap+2 + T * (-0x1.1c98643a78c6ap-11 + T * (0x1.18be22e62f026p-16 + T * (-0x1.72b101d35ae59p-26 + T * 0x1.2f72fba30b7c2p-37)))), cpm);
      cpm = fma(s[8] * irho, 0x1.3f5713b5bf6a1p+9 * (0x1.beb24fde64a4cp+1 + T * (0x1.5390f0ed10ec5p-12 + T * (-0x1.c5628dbdf8e58p-20 + T * (0x1.b29b14b88d49cp-29 + T * -0x1.8bc782bbe23bbp-40)))), cpm);
      cpm = fma(s[9] * irho, 0x1.28d5af07bfe7ep+8 * (0x1.ca2e271a4b2fdp+1 + T * (-0x1.400048c1ba1b0p-11 + T * (0x1.10f2f2ddb1673p-20 + T * (0x1.f2a1bae3bf93ap-31 + T * -0x1.fd254e88ba403p-41)))), cpm);
      cpm = fma(s[10] * irho, 0x1.2863e90ff9724p+9 * (0x1.e19f746480de1p+1 + T * (0x1.fbf7d158743a2p-11 + T * (0x1.771ffa66e83e0p-19 + T * (-0x1.08a1f3bb46844p-28 + T * 0x1.daf7390cac908p-40)))), cpm);
      cpm = fma(s[11] * irho, 0x1.1e860685553efp+8 * (0x1.0e27e8a748d9cp+2 + T * (-0x1.a9301251f436fp-9 + T * (0x1.ce60d2a2b7dfep-17 + T * (-0x1.c97ac8618dbf3p-27 + T * 0x1.313cda197894cp-38)))), cpm);
      cpm = fma(s[12] * irho, 0x1.2863e90ff9724p+9 * (0x1.0cb5ee035346ap+2 + T * (-0x1.36326518bab75p-9 + T * (0x1.14409b5702698p-17 + T * (-0x1.cb9b5a07323d1p-28 + T * 0x1.1179431daea17p-39)))), cpm);
      cpm = fma(s[13] * irho, 0x1.148494a2b9d3dp+9 * (0x1.d63835d17324cp+1 + T * (0x1.079458000b018p-9 + T * (0x1.808c67bee451fp-18 + T * (-0x1.d82ef9cab9cf9p-28 + T * 0x1.66041ea7cf186p-39)))), cpm);
      cpm = fma(s[14] * irho, 0x1.14e7994e1a3f4p+8 * (0x1.32cc5c2ed4ffap+2 + T * (-0x1.44ad209405144p-7 + T * (0x1.391462ecfccf9p-15 + T * (-0x1.45cdb600576d1p-25 + T * 0x1.cfa240d78baa9p-37)))), cpm);
      cpm = fma(s[15] * irho, 0x1.03249374bc6a8p+9 * (0x1.4997920d33445p+2 + T * (-0x1.bff87b6cd6efap-7 + T * (0x1.9c8d5fdb7d96ep-15 + T * (-0x1.a0641e640b81dp-25 + T * 0x1.254048a7f227ep-36)))), cpm);
      cpm = fma(s[16] * irho, 0x1.79d6b356da017p+7 * (0x1.2daac1343d496p+1 + T * (0x1.266842a5bf315p-7 + T * (-0x1.de0de0090effep-18 + T * (0x1.51fd10511d1a8p-29 + T * -0x1.43952648a136cp-43)))), cpm);
      cpm = fma(s[17] * irho, 0x1.0be922424a277p+8 * (0x1.ee93ebafbbefep+1 + T * (0x1.6ec96e6bebfdfp-8 + T * (0x1.8e23514e314c1p-18 + T * (-0x1.672b5483bb261p-27 + T * 0x1.337d06dd584f1p-38)))), cpm);
      cpm = fma(s[18] * irho, 0x1.0be922424a277p+8 * (0x1.0d9817b95a294p+1 + T * (0x1.d8f25f83733c9p-8 + T * (0x1.664240277b618p-18 + T * (-0x1.fafcbebd8fc7ap-28 + T * 0x1.241dbb3bc1290p-39)))), cpm);
      cpm = fma(s[19] * irho, 0x1.037b88a8b08ddp+8 * (0x1.6dc90b8ca6163p+2 + T * (-0x1.f316286598c3ep-7 + T * (0x1.11a755e8b7abap-14 + T * (-0x1.314a0b40b1447p-24 + T * 0x1.cbc6ca94c4677p-36)))), cpm);
      cpm = fma(s[20] * irho, 0x1.4c3397bb73083p+8 * (0x1.71e04a987f933p+1 + T * (0x1.b76ae82ebca6cp-7 + T * (-0x1.ddc391c23021ap-16 + T * (0x1.fa727902a68efp-26 + T * -0x1.80ad12085942bp-37)))), cpm);
      cpm = fma(s[21] * irho, 0x1.3f5713ad5bee4p+8 * (0x1.9e0b72c73f3bap-1 + T * (0x1.7ec17f28e481ap-6 + T * (-0x1.29f09105c533cp-15 + T * (0x1.e14c5845a203fp-26 + T * -0x1.2b17c43e837e8p-37)))), cpm);
      cpm = fma(s[22] * irho, 0x1.954cff43419e3p+7 * (0x1.203868265a06ep+1 + T * (0x1.2142867388492p-6 + T * (-0x1.8e1bb67756fd6p-16 + T * (0x1.28cb9772e0568p-26 + T * -0x1.64859c0d2ee1dp-38)))), cpm);
      cpm = fma(s[23] * irho, 0x1.33700096feb4ap+8 * (0x1.9b3219c31fa4ep+1 + T * (0x1.8d17f1df63fcdp-10 + T * (0x1.b2e198409699cp-16 + T * (-0x1.3339cad4b897fp-25 + T * 0x1.02dedc9720552p-36)))), cpm);
      cpm = fma(s[24] * irho, 0x1.8b94f63800219p+7 * (0x1.116315790e08dp+1 + T * (0x1.28dc0ec708b6bp-6 + T * (-0x1.23d5df074d80ap-16 + T * (0x1.410e7ab1ff68dp-27 + T * -0x1.1b86c153f96acp-39)))), cpm);
      cpm = fma(s[25] * irho, 0x1.2863e90ff9724p+8 * (0x1.fac71d356ff96p+1 + T * (-0x1.f0244a6c1abf8p-8 + T * (0x1.defb3b4522b25p-15 + T * (-0x1.2908fcd07cb16p-24 + T * 0x1.dac91dbd28c88p-36)))), cpm);
      cpm = fma(s[26] * irho, 0x1.1e1c0389f83bep+8 * (0x1.139d223a3c91dp+2 + T * (-0x1.125f4e7e42173p-8 + T * (0x1.a1089ad91c191p-15 + T * (-0x1.0152aabf3f38cp-24 + T * 0x1.958406c58ed2fp-36)))), cpm);
      cpm = fma(s[27] * irho, 0x1.148494a2b9d3dp+8 * (0x1.12a6b4b528ec3p+2 + T * (-0x1.688c91f95b2dfp-8 + T * (0x1.f6d86463b6ba0p-15 + T * (-0x1.3048b11b68ad6p-24 + T * 0x1.d8ad50563705bp-36)))), cpm);
      cpm = fma(s[28] * irho, 0x1.cd7f5ff609dd0p+8 * (0x1.0cb686e536fbfp+2 + T * (-0x1.0aeb63b84c925p-9 + T * (0x1.b593a7c039b70p-18 + T * (-0x1.7921667072d59p-28 + T * 0x1.f2c47bce627b1p-40)))), cpm);
      cpm = fma(s[29] * irho, 0x1.a04215336deb9p+7 * (0x1.4000000000000p+1 + T * (0.0 + T * (0.0 + T * (0.0 + T * 0.0)))), cpm);
      cpm = fma(s[30] * irho, 0x1.5a24731d2e0e3p+9 * (0x1.46f15252b32b4p+1 + T * (-0x1.51282024e7f51p-12 + T * (0x1.89f3a3624c78ep-21 + T * (-0x1.928ce62f9cb00p-31 + T * 0x1.2c13939e39b46p-42)))), cpm);
      cpm = fma(s[31] * irho, 0x1.8b94f63800219p+7 * (0x1.3e0c2d34ec70dp+0 + T * (0x1.fd1641c705f4ap-6 + T * (-0x1.aab3c237df3eep-15 + T * (0x1.728b8de31e2a5p-25 + T * -0x1.ed183d9a14087p-37)))), cpm);
      cpm = fma(s[32] * irho, 0x1.825174a3400b9p+7 * (0x1.b45c24c404a73p+1 + T * (0x1.5fe1b0115dd40p-7 + T * (0x1.fbbe572a5fd07p-20 + T * (-0x1.ebef1fbb3686fp-28 + T * 0x1.938c6ea0bdd8cp-39)))), cpm);
      cpm = fma(s[33] * irho, 0x1.797a7aa68f4b6p+7 * (0x1.2eaf76e6106abp+2 + T * (-0x1.a28ce427d2efep-9 + T * (0x1.8ec0772eb57cep-15 + T * (-0x1.ed90d262d7aa3p-25 + T * 0x1.81d0f2a50dc3bp-36)))), cpm);
      cpm = fma(s[34] * irho, 0x1.791e6f0cfe154p+7 * (0x1.ddfac3d6032c6p-1 + T * (0x1.b0f0b7a76578fp-6 + T * (0x1.99c3cfee1d154p-18 + T * (-0x1.79921013a4d49p-26 + T * 0x1.4ec6d3fc774f1p-37)))), cpm);
      cpm = fma(s[35] * irho, 0x1.81f10d173fb7ap+7 * (0x1.0d327faf0cc86p+0 + T * (0x1.a9da4403baf59p-6 + T * (0x1.3f720861c2c5bp-19 + T * (-0x1.50e3cbe90afe8p-26 + T * 0x1.49cab4118eabap-37)))), cpm);
    }
    rates(C, T, P, cd);
    f[0] = cd[0] * 0x1.c051ec0000000p+4;
    f[1] = cd[1] * 0x1.0000000000000p+4;
    f[2] = cd[2] * 0x1.0000000000000p+5;
    f[3] = cd[3] * 0x1.020c4a0000000p+0;
    f[4] = cd[4] * 0x1.1020c40000000p+4;
    f[5] = cd[5] * 0x1.020c4a0000000p+1;
    f[6] = cd[6] * 0x1.0810620000000p+5;
    f[7] = cd[7] * 0x1.1020c40000000p+5;
    f[8] = cd[8] * 0x1.a093740000000p+3;
    f[9] = cd[9] * 0x1.c028f60000000p+4;
    f[10] = cd[10] * 0x1.c0d4fe0000000p+3;
    f[11] = cd[11] * 0x1.d049ba0000000p+4;
    f[12] = cd[12] * 0x1.c0d4fe0000000p+3;
    f[13] = cd[13] * 0x1.e116880000000p+3;
    f[14] = cd[14] * 0x1.e06a7e0000000p+4;
    f[15] = cd[15] * 0x1.00ac080000000p+4;
    f[16] = cd[16] * 0x1.60147a0000000p+5;
    f[17] = cd[17] * 0x1.f08b440000000p+4;
    f[18] = cd[18] * 0x1.f08b440000000p+4;
    f[19] = cd[19] * 0x1.0056040000000p+5;
    f[20] = cd[20] * 0x1.9072b00000000p+4;
    f[21] = cd[21] * 0x1.a093740000000p+4;
    f[22] = cd[22] * 0x1.4839580000000p+5;
    f[23] = cd[23] * 0x1.b0b43a0000000p+4;
    f[24] = cd[24] * 0x1.5049ba0000000p+5;
    f[25] = cd[25] * 0x1.c0d4fe0000000p+4;
    f[26] = cd[26] * 0x1.d0f5c20000000p+4;
    f[27] = cd[27] * 0x1.e116880000000p+4;
    f[28] = cd[28] * 0x1.20418a0000000p+4;
    f[29] = cd[29] * 0x1.3f95820000000p+5;
    f[30] = cd[30] * 0x1.8051ec0000000p+3;
    f[31] = cd[31] * 0x1.5049ba0000000p+5;
    f[32] = cd[32] * 0x1.585a1c0000000p+5;
    f[33] = cd[33] * 0x1.606a7e0000000p+5;
    f[34] = cd[34] * 0x1.60c0840000000p+5;
    f[35] = cd[35] * 0x1.58b0200000000p+5;
    double tmp = 0.0;
    if (hi) {
      tmp = fma(-(0x1.28ba9057d1783p+8 * (T * (0x1.769c23b7952d2p+1 + T * (0x1.86106ec5d7fc6p-11 + T * (-0x1.96ee5424b7af6p-23 + T * (0x1.bc128a9b8a724p-36 + T * -0x1.854ddeba4197bp-50)))) + -0x1.cd661b089a027p+9)), f[0], tmp);
      tmp = fma(-(0x1.03d2b851eb852p+9 * (T * (0x1.48e2c7b5e1a3dp+1 + T * (-0x1.689a0073e4c12p-15 + T * (0x1.e0722e91f065fp-27 + T * (-0x1.607823b4427e2p-39 + T * 0x1.1b3c369230ddcp-52)))) + 0x1.c88650ff97247p+14)), f[1], tmp);
      tmp = fma(-(0x1.03d2b851eb852p+8 * (T * (0x1.a42a332f575b8p+1 + T * (0x1.84c851ecf574dp-11 + T * (-0x1.0f496e2f6b32bp-22 + T * (0x1.cca17066bf423p-35 + T * -0x1.3852c0eebb013p-48)))) + -0x1.101d4b48d3ae7p+10)), f[2], tmp);
      tmp = fma(-(0x1.01c2d34acaff7p+13 * (T * (0x1.40000015798eep+1 + T * (-0x1.961a6ea91e1b0p-37 + T * (0x1.840f104982ce0p-48 + T * (-0x1.5d647fca8f878p-60 + T * 0x1.e1d3b0ee8129dp-74)))) + 0x1.8e06a3bcd35a8p+14)), f[3], tmp);
      tmp = fma(-(0x1.e8d949731098dp+8 * (T * (0x1.8be3be406d029p+1 + T * (0x1.1f88fd8e1440ep-12 + T * (0x1.6a39500d21114p-25 + T * (-0x1.82ca91827ab6dp-36 + T * 0x1.526b0ac38c4c6p-49)))) + 0x1.e2550624dd2f2p+11)), f[4], tmp);
      tmp = fma(-(0x1.01c2d350092cdp+12 * (T * (0x1.ab2bf6fecf7e5p+1 + T * (-0x1.9e6b00c08fd91p-16 + T * (0x1.65866c34c762ap-23 + T * (-0x1.8adee4a4b6baep-35 + T * 0x1.2099318342be3p-48)))) + -0x1.db14578e5c4ebp+9)), f[5], tmp);
      tmp = fma(-(0x1.f7c6fae7924afp+7 * (T * (0x1.0119fbbf289f6p+2 + T * (0x1.2593e454221e1p-10 + T * (-0x1.c597157493eb4p-23 + T * (0x1.f675fa32f618cp-36 + T * -0x1.370671f4bb474p-49)))) + 0x1.bf6d462c343b7p+6)), f[6], tmp);
      tmp = fma(-(0x1.e8d94983d7907p+7 * (T * (0x1.0a8f681d1fcb7p+2 + T * (0x1.41abe4bc5704bp-9 + T * (-0x1.544474260f258p-21 + T * (0x1.981f91177d524p-34 + T * -0x1.9eeb6a97eb6fbp-48)))) + -0x1.1717269ad42c4p+14)), f[7], tmp);
      tmp = fma(-(0x1.3f5713b5bf6a1p+9 * (T * (0x1.70718843050d6p+1 + T * (0x1.fd09d405d0756p-12 + T * (0x1.9d97c8efd3589p-25 + T * (-0x1.1f62b7f778ce2p-35 + T * 0x1.fb83a7106ba7cp-49)))) + 0x1.15646fb7e9100p+16)), f[8], tmp);
      tmp = fma(-(0x1.28d5af07bfe7ep+8 * (T * (0x1.5b8b33bac2892p+1 + T * (0x1.0e56efcdc62d9p-10 + T * (-0x1.657e6113731d3p-22 + T * (0x1.f9e45483ed15bp-35 + T * -0x1.257cbef78f170p-48)))) + -0x1.ba3efaacd9e84p+13)), f[9], tmp);
      tmp = fma(-(0x1.2863e90ff9724p+9 * (T * (0x1.6fe28bbb5f921p+1 + T * (0x1.df4030068403dp-10 + T * (-0x1.f8480a32a419ap-22 + T * (0x1.1e12084ded447p-34 + T * -0x1.0e8b3f67fea4fp-48)))) + 0x1.696f353f7ced9p+15)), f[10], tmp);
      tmp = fma(-(0x1.1e860685553efp+8 * (T * (0x1.62d69c2e745cap+1 + T * (0x1.44dbe8babc438p-9 + T * (-0x1.bc9c59a08596ap-21 + T * (0x1.43e5262ed5e8fp-33 + T * -0x1.806efc81153b4p-47)))) + 0x1.f57d617c1bda5p+11)), f[11], tmp);
      tmp = fma(-(0x1.2863e90ff9724p+9 * (T * (0x1.256183d389aa6p+1 + T * (0x1.3120cfa66c760p-9 + T * (-0x1.680c0911ecdbfp-21 + T * (0x1.cb7e14e4de1f4p-34 + T * -0x1.e9953783e1eedp-48)))) + 0x1.8ddbffd8adabap+15)), f[12], tmp);
      tmp = fma(-(0x1.148494a2b9d3dp+9 * (T * (0x1.249265f3a4d2ep+1 + T * (0x1.da795f45c2785p-9 + T * (-0x1.0b48fa9ba4676p-20 + T * (0x1.477b292040de5p-33 + T * -0x1.509ec68687becp-47)))) + 0x1.061e5652bd3c3p+14)), f[13], tmp);
      tmp = fma(-(0x1.14e7994e1a3f4p+8 * (T * (0x1.c2bc95c7fddb1p+0 + T * (0x1.2d77335291c21p-8 + T * (-0x1.8bb9fb006a417p-20 + T * (0x1.14a3f4fe94722p-32 + T * -0x1.3e714b400a419p-46)))) + -0x1.b55ea88ce703bp+13)), f[14], tmp);
      tmp = fma(-(0x1.03249374bc6a8p+9 * (T * (0x1.32977b314eac9p-4 + T * (0x1.b6cb6711ca116p-8 + T * (-0x1.007bd5b5d2422p-19 + T * (0x1.5027b8a366174p-32 + T * -0x1.6ed3f97ad9a01p-46)))) + -0x1.27e2c1b866e44p+13)), f[15], tmp);
      tmp = fma(-(0x1.79d6b356da017p+7 * (T * (0x1.edc1423f95973p+1 + T * (0x1.214cd7e62db66p-9 + T * (-0x1.8c5b3dc67eba3p-21 + T * (0x1.1fcab1b9912a3p-33 + T * -0x1.542c2854e86a3p-47)))) + -0x1.7cee54fdf3b64p+15)), f[16], tmp);
      tmp = fma(-(0x1.0be922424a277p+8 * (T * (0x1.d8a944f2ce3e4p+1 + T * (0x1.1b4df55c881e2p-8 + T * (-0x1.4fa2825a8a1ddp-20 + T * (0x1.b0c96ce8203e2p-33 + T * -0x1.d3552229febefp-47)))) + -0x1.9550335d249e4p+11)), f[17], tmp);
      tmp = fma(-(0x1.0be922424a277p+8 * (T * (0x1.e2a98aa8650e7p+1 + T * (0x1.01eee717c07fdp-8 + T * (-0x1.db60e102b316bp-21 + T * (0x1.b1b1dcc557332p-34 + T * -0x1.3075c5faa9762p-48)))) + 0x1.ff54801f75105p+6)), f[18], tmp);
      tmp = fma(-(0x1.037b88a8b08ddp+8 * (T * (0x1.ca2a4c2ed7aedp+0 + T * (0x1.cdd39bbea4fb5p-8 + T * (-0x1.1cc401d83630dp-19 + T * (0x1.7bcd41e9ad83ep-32 + T * -0x1.a5c0fef86370dp-46)))) + -0x1.8c7b7fb15b574p+14)), f[19], tmp);
      tmp = fma(-(0x1.4c3397bb73083p+8 * (T * (0x1.957aaf1dba502p+1 + T * (0x1.377101463a6fcp-9 + T * (-0x1.48e6585748e57p-21 + T * (0x1.4e75f1b05c789p-34 + T * -0x1.fed6b3b564915p-49)))) + 0x1.063110a3d70a4p+16)), f[20], tmp);
      tmp = fma(-(0x1.3f5713ad5bee4p+8 * (T * (0x1.0971c7ee6bae0p+2 + T * (0x1.86b42b3f9ab1ep-9 + T * (-0x1.a8a7da8ef5fe7p-21 + T * (0x1.00f66a44e90d0p-33 + T * -0x1.044c229f7f34fp-47)))) + 0x1.953fff2e48e8ap+14)), f[21], tmp);
      tmp = fma(-(0x1.954cff43419e3p+7 * (T * (0x1.683486198a14cp+2 + T * (0x1.0bbca21f5e9bfp-9 + T * (-0x1.1d28ea5e6fd95p-21 + T * (0x1.3abf2c56d8d5fp-34 + T * -0x1.17b2431182340p-48)))) + 0x1.2dfcdc28f5c29p+14)), f[22], tmp);
      tmp = fma(-(0x1.33700096feb4ap+8 * (T * (0x1.8224031487768p+1 + T * (0x1.52803e497ede9p-8 + T * (-0x1.a2d53f48cbb22p-20 + T * (0x1.17b98c3c9686ep-32 + T * -0x1.36c974de2fce9p-46)))) + 0x1.0e69bf6fd21ffp+15)), f[23], tmp);
      tmp = fma(-(0x1.8b94f63800219p+7 * (T * (0x1.20b91864fbad3p+2 + T * (0x1.2707a6468c0fap-8 + T * (-0x1.75123eb3ba5c4p-20 + T * (0x1.fb9d6149efe38p-33 + T * -0x1.1e5ee25ffae6bp-46)))) + -0x1.d7f0d989df117p+12)), f[24], tmp);
      tmp = fma(-(0x1.2863e90ff9724p+8 * (T * (0x1.049f4a5d9c3d6p+1 + T * (0x1.dfe6a5720731ep-8 + T * (-0x1.2c3c3485b62c8p-19 + T * (0x1.94aeec15226e0p-32 + T * -0x1.c4e760753f615p-46)))) + 0x1.34be2da122fadp+12)), f[25], tmp);
      tmp = fma(-(0x1.1e1c0389f83bep+8 * (T * (0x1.f4645cf6d1024p+0 + T * (0x1.1d0972c8defc6p-7 + T * (-0x1.651c92fac6c2cp-19 + T * (0x1.e1a27ccaa5e06p-32 + T * -0x1.0d91ff12db09fp-45)))) + 0x1.91cc28f5c28f6p+13)), f[26], tmp);
      tmp = fma(-(0x1.148494a2b9d3dp+8 * (T * (0x1.1266d373affb0p+0 + T * (0x1.634a9b006255bp-7 + T * (-0x1.c089bdb6616a1p-19 + T * (0x1.304e6c1f3af79p-31 + T * -0x1.56475dfc0f594p-45)))) + -0x1.651325460aa65p+13)), f[27], tmp);
      tmp = fma(-(0x1.cd7f5ff609dd0p+8 * (T * (0x1.8459ddac6e07ap+1 + T * (0x1.1d553f9364039p-10 + T * (-0x1.d5ca6d6fbef3fp-25 + T * (-0x1.aacb905b9d982p-36 + T * 0x1.e4ce6d148b330p-49)))) + -0x1.d4d1303afb7e9p+14)), f[28], tmp);
      tmp = fma(-(0x1.a04215336deb9p+7 * (T * (0x1.4000000000000p+1 + T * (0.0 + T * (0.0 + T * (0.0 + T * 0.0)))) + -0x1.74b0000000000p+9)), f[29], tmp);
      tmp = fma(-(0x1.5a24731d2e0e3p+9 * (T * (0x1.3f0fc61badb08p+1 + T * (0x1.928f7063e1320p-16 + T * (-0x1.9ecca316c19acp-26 + T * (0x1.493ad8d3ca4a8p-37 + T * -0x1.18e5865166a28p-50)))) + 0x1.4dcb4b98c7e28p+16)), f[30], tmp);
      tmp = fma(-(0x1.8b94f63800219p+7 * (T * (0x1.7b200416e5f59p+2 + T * (0x1.bd24e4100a643p-9 + T * (-0x1.cb2d8a1cf4050p-21 + T * (0x1.eea583fa736bdp-34 + T * -0x1.af7b79e42769ap-48)))) + 0x1.c60a04189374cp+12)), f[31], tmp);
      tmp = fma(-(0x1.825174a3400b9p+7 * (T * (0x1.7e7160956c0d7p+2 + T * (0x1.0a6c5738986f4p-8 + T * (-0x1.eafd9a8d0705ep-21 + T * (0x1.bf88df5305066p-34 + T * -0x1.3998db7e70d3ep-48)))) + 0x1.ea52617c1bda5p+8)), f[32], tmp);
      tmp = fma(-(0x1.797a7aa68f4b6p+7 * (T * (0x1.59dcf38b7d772p+2 + T * (0x1.80242581cd52bp-8 + T * (-0x1.7a2a05927a704p-20 + T * (0x1.77e1aba8e49a3p-33 + T * -0x1.2753ba556825fp-47)))) + -0x1.61047ced91687p+14)), f[33], tmp);
      tmp = fma(-(0x1.791e6f0cfe154p+7 * (T * (0x1.e22f4c1de5c41p+2 + T * (0x1.3533e853aabbcp-7 + T * (-0x1.18990810740d6p-19 + T * (0x1.f6e487f8d81b8p-33 + T * -0x1.58b5a95d75eb1p-47)))) + -0x1.014e10624dd2fp+14)), f[34], tmp);
      tmp = fma(-(0x1.81f10d173fb7ap+7 * (T * (0x1.ecf903f7dc451p+2 + T * (0x1.06de43cb39826p-7 + T * (-0x1.d8be5fcb25bf4p-20 + T * (0x1.a374b81e9310cp-33 + T * -0x1.1bd9f02a1e858p-47)))) + 0x1.0353780346dc6p+13)), f[35], tmp);
    } else {
      tmp = fma(-(0x1.28ba9057d1783p+8 * (T * (0x1.a63b0c4588a05p+1 + T * (0x1.712969da04050p-11 + T * (-0x1.629f839620fc6p-20 + T * (0x1.83ae94da0fe59p-30 + T * -0x1.13441e6a0b3dfp-41)))) + -0x1.fe732fec56d5dp+9)), f[0], tmp);
      tmp = fma(-(0x1.03d2b851eb852p+9 * (T * (0x1.9589c6bdbf12dp+1 + T * (-0x1.add3ae5787a18p-10 + T * (0x1.2934a57c4d958p-19 + T * (-0x1.a51e14d5c0503p-30 + T * 0x1.dbba8a635ed80p-42)))) + 0x1.c709096bb98c8p+14)), f[1], tmp);
      tmp = fma(-(0x1.03d2b851eb852p+8 * (T * (0x1.e42787ae5fa45p+1 + T * (-0x1.88c9b66c8c0dfp-10 + T * (0x1.b88f92cda255fp-19 + T * (-0x1.4ca5927516966p-29 + T * 0x1.6d361ad59bca4p-41)))) + -0x1.09fc63497b741p+10)), f[2], tmp);
      tmp = fma(-(0x1.01c2d34acaff7p+13 * (T * (0x1.4000000000000p+1 + T * (0x1.8d112bf5fb7e0p-42 + T * (-0x1.7f85eab504006p-51 + T * (0x1.538a620b2373fp-61 + T * -0x1.c09fb31fd8141p-73)))) + 0x1.8e06a3bcd35a8p+14)), f[3], tmp);
      tmp = fma(-(0x1.e8d949731098dp+8 * (T * (0x1.fefa5c927d1abp+1 + T * (-0x1.3abed86e71c7dp-10 + T * (0x1.9d34c5287c942p-20 + T * (-0x1.0ab59e9c18f85p-30 + T * 0x1.332bdbce74b0fp-42)))) + 0x1.c3e293f290abbp+11)), f[4], tmp);
      tmp = fma(-(0x1.01c2d350092cdp+12 * (T * (0x1.2c130ac9b2911p+1 + T * (0x1.058175caab342p-8 + T * (-0x1.b3b80759749d1p-18 + T * (0x1.5a4c582f87e3dp-28 + T * -0x1.9f3d0eb996c74p-40)))) + -0x1.caf7b3bfb58d1p+9)), f[5], tmp);
      tmp = fma(-(0x1.f7c6fae7924afp+7 * (T * (0x1.1350a899bcaa1p+2 + T * (-0x1.373d053b75995p-9 + T * (0x1.d94d8bd675c95p-18 + T * (-0x1.a110b0905e0fcp-28 + T * 0x1.058dba115721ap-39)))) + 0x1.26cedbb59ddc2p+8)), f[6], tmp);
      tmp = fma(-(0x1.e8d94983d7907p+7 * (T * (0x1.11abd48f63e0ap+2 + T * (-0x1.1c986431acf9ep-12 + T * (0x1.7652d932e9587p-18 + T * (-0x1.72b101cd97284p-28 + T * 0x1.e584c5e48fadep-40)))) + -0x1.149a541205bc0p+14)), f[7], tmp);
      tmp = fma(-(0x1.3f5713b5bf6a1p+9 * (T * (0x1.beb24fde64a4cp+1 + T * (0x1.5390f0fea885dp-13 + T * (-0x1.2e41b3d0faa66p-21 + T * (0x1.b29b14b3f0b25p-31 + T * -0x1.3c9f9bc981c95p-42)))) + 0x1.148d4b1c432cap+16)), f[8], tmp);
      tmp = fma(-(0x1.28d5af07bfe7ep+8 * (T * (0x1.ca2e271a4b2fdp+1 + T * (-0x1.400048c1ba1b0p-12 + T * (0x1.6bee992797344p-22 + T * (0x1.f2a1bae3bf93ap-33 + T * -0x1.97510ba823483p-43)))) + -0x1.c040b020c49bap+13)), f[9], tmp);
      tmp = fma(-(0x1.2863e90ff9724p+9 * (T * (0x1.e19f746480de1p+1 + T * (0x1.fbf7d1614006ep-12 + T * (0x1.f42aa330dfb56p-21 + T * (-0x1.08a1f3bd94cffp-30 + T * 0x1.7bf8fa708a0d3p-42)))) + 0x1.67681487fcb92p+15)), f[10], tmp);
      tmp = fma(-(0x1.1e860685553efp+8 * (T * (0x1.0e27e8a748d9cp+2 + T * (-0x1.a9301251f436fp-10 + T * (0x1.34408c703b59dp-18 + T * (-0x1.c97ac86d1539dp-29 + T * 0x1.e8615cf58dbadp-41)))) + 0x1.dff21426fe719p+11)), f[11], tmp);
      tmp = fma(-(0x1.2863e90ff9724p+9 * (T * (0x1.0cb5ee035346ap+2 + T * (-0x1.3632652eb8373p-10 + T * (0x1.7056246c81ae3p-19 + T * (-0x1.cb9b59fbaac26p-30 + T * 0x1.b58ed1c91768bp-42)))) + 0x1.8a81a1f212d77p+15)), f[12], tmp);
      tmp = fma(-(0x1.148494a2b9d3dp+9 * (T * (0x1.d63835d17324cp+1 + T * (0x1.0794581608816p-10 + T * (0x1.005d9a77c1582p-19 + T * (-0x1.d82ef9bf3254fp-30 + T * 0x1.1e69b21fd8e05p-41)))) + 0x1.00f3fec56d5d0p+14)), f[13], tmp);
      tmp = fma(-(0x1.14e7994e1a3f4p+8 * (T * (0x1.32cc5c2ed4ffap+2 + T * (-0x1.44ad208e85b45p-8 + T * (0x1.a17083d3e2933p-17 + T * (-0x1.45cdb5fd758e7p-27 + T * 0x1.72e833dfa2eeep-39)))) + -0x1.bf27a7525460bp+13)), f[14], tmp);
      tmp = fma(-(0x1.03249374bc6a8p+9 * (T * (0x1.4997920d33445p+2 + T * (-0x1.bff87b6cd6efap-8 + T * (0x1.1308ea9253b9fp-16 + T * (-0x1.a0641e80de346p-27 + T * 0x1.d533a7731d0cap-39)))) + -0x1.40352e48e8a72p+13)), f[15], tmp);
      tmp = fma(-(0x1.79d6b356da017p+7 * (T * (0x1.2daac1343d496p+1 + T * (0x1.266842ab3e914p-8 + T * (-0x1.3eb3eab83633cp-19 + T * (0x1.51fd10511d1a8p-31 + T * -0x1.02ddb83a1a924p-45)))) + -0x1.79e7f07c84b5ep+15)), f[16], tmp);
      tmp = fma(-(0x1.0be922424a277p+8 * (T * (0x1.ee93ebafbbefep+1 + T * (0x1.6ec96e6bebfdfp-9 + T * (0x1.096ce0e64d114p-19 + T * (-0x1.672b5483bb261p-29 + T * 0x1.ebfb3e2ef3b1bp-41)))) + -0x1.8f3d3cc8de2acp+11)), f[17], tmp);
      tmp = fma(-(0x1.0be922424a277p+8 * (T * (0x1.0d9817b95a294p+1 + T * (0x1.d8f25f83733c9p-9 + T * (0x1.ddadaaee523f0p-20 + T * (-0x1.fafcbebd8fc7ap-30 + T * 0x1.d362c52c6841ap-42)))) + 0x1.e94cf0d844d01p+9)), f[18], tmp);
      tmp = fma(-(0x1.037b88a8b08ddp+8 * (T * (0x1.6dc90b8ca6163p+2 + T * (-0x1.f316286598c3ep-8 + T * (0x1.6cdf1d364a3a3p-16 + T * (-0x1.314a0b397c97dp-26 + T * 0x1.6fd23baa36b93p-38)))) + -0x1.90ab0ff972474p+14)), f[19], tmp);
      tmp = fma(-(0x1.4c3397bb73083p+8 * (T * (0x1.71e04a987f933p+1 + T * (0x1.b76ae82ebca6cp-8 + T * (-0x1.3e82612c20167p-17 + T * (0x1.fa7279086a4c4p-28 + T * -0x1.33bda806adcefp-39)))) + 0x1.051764a8c154dp+16)), f[20], tmp);
      tmp = fma(-(0x1.3f5713ad5bee4p+8 * (T * (0x1.9e0b72c73f3bap-1 + T * (0x1.7ec17f4461617p-7 + T * (-0x1.8d40c15d06efbp-17 + T * (0x1.e14c583fde46ap-28 + T * -0x1.de8c6d3a443e1p-40)))) + 0x1.9cf3ec3c9eeccp+14)), f[21], tmp);
      tmp = fma(-(0x1.954cff43419e3p+7 * (T * (0x1.203868265a06ep+1 + T * (0x1.2142867388492p-7 + T * (-0x1.0967cef8599c0p-17 + T * (0x1.28cb9772e0568p-28 + T * -0x1.1d37b00a8be7dp-40)))) + 0x1.396dcbc6a7efap+14)), f[22], tmp);
      tmp = fma(-(0x1.33700096feb4ap+8 * (T * (0x1.9b3219c31fa4ep+1 + T * (0x1.8d17f1df63fcdp-11 + T * (0x1.21ebbad3d9599p-17 + T * (-0x1.3339cad1d6b94p-27 + T * 0x1.9e3160f1cd550p-39)))) + 0x1.1057b18fc5048p+15)), f[23], tmp);
      tmp = fma(-(0x1.8b94f63800219p+7 * (T * (0x1.116315790e08dp+1 + T * (0x1.28dc0ec708b6bp-7 + T * (-0x1.851d295b513c4p-18 + T * (0x1.410e7ab1ff68dp-29 + T * -0x1.c5a468865bde0p-42)))) + -0x1.b82eb04ab606bp+12)), f[24], tmp);
      tmp = fma(-(0x1.2863e90ff9724p+8 * (T * (0x1.fac71d356ff96p+1 + T * (-0x1.f0244a77197f7p-9 + T * (0x1.3f52277a0a8b7p-16 + T * (-0x1.2908fcc94804cp-26 + T * 0x1.7bd417ca8706cp-38)))) + 0x1.3e1c6a35935fcp+12)), f[25], tmp);
      tmp = fma(-(0x1.1e1c0389f83bep+8 * (T * (0x1.139d223a3c91dp+2 + T * (-0x1.125f4e7e42173p-9 + T * (0x1.1605bc90bd661p-16 + T * (-0x1.0152aab0d5df8p-26 + T * 0x1.44699f0472426p-38)))) + 0x1.914d03126e979p+13)), f[26], tmp);
      tmp = fma(-(0x1.148494a2b9d3dp+8 * (T * (0x1.12a6b4b528ec3p+2 + T * (-0x1.688c91f95b2dfp-9 + T * (0x1.4f3aeda131122p-16 + T * (-0x1.3048b1143400cp-26 + T * 0x1.7a244044f8d16p-38)))) + -0x1.6811a4dd2f1aap+13)), f[27], tmp);
      tmp = fma(-(0x1.cd7f5ff609dd0p+8 * (T * (0x1.0cb686e536fbfp+2 + T * (-0x1.0aeb63b84c925p-10 + T * (0x1.23b7c52ad124bp-19 + T * (-0x1.7921668781cadp-30 + T * 0x1.8f03963eb52f4p-42)))) + -0x1.d956e8240b780p+14)), f[28], tmp);
      tmp = fma(-(0x1.a04215336deb9p+7 * (T * (0x1.4000000000000p+1 + T * (0.0 + T * (0.0 + T * (0.0 + T * 0.0)))) + -0x1.74b0000000000p+9)), f[29], tmp);
      tmp = fma(-(0x1.5a24731d2e0e3p+9 * (T * (0x1.46f15252b32b4p+1 + T * (-0x1.51282024e7f51p-13 + T * (0x1.06a26cec32fb4p-22 + T * (-0x1.928ce62663812p-33 + T * 0x1.e01f5296c2ba3p-45)))) + 0x1.4dc3e219652bdp+16)), f[30], tmp);
      tmp = fma(-(0x1.8b94f63800219p+7 * (T * (0x1.3e0c2d34ec70dp+0 + T * (0x1.fd1641c705f4ap-7 + T * (-0x1.1c77d6c6883e7p-16 + T * (0x1.728b8dfff0dcep-27 + T * -0x1.8a79cae1a9a06p-39)))) + 0x1.f5f9d42c3c9efp+12)), f[31], tmp);
      tmp = fma(-(0x1.825174a3400b9p+7 * (T * (0x1.b45c24c404a73p+1 + T * (0x1.5fe1b0115dd40p-8 + T * (0x1.527ee4c3e9edbp-21 + T * (-0x1.ebef1fbb3686fp-30 + T * 0x1.42d6bee6fe470p-41)))) + 0x1.7c5e809d49518p+10)), f[32], tmp);
      tmp = fma(-(0x1.797a7aa68f4b6p+7 * (T * (0x1.2eaf76e6106abp+2 + T * (-0x1.a28ce427d2efep-10 + T * (0x1.09d5a4d3303ebp-16 + T * (-0x1.ed90d24604f7ap-27 + T * 0x1.34a728840b02fp-38)))) + -0x1.511383126e979p+14)), f[33], tmp);
      tmp = fma(-(0x1.791e6f0cfe154p+7 * (T * (0x1.ddfac3d6032c6p-1 + T * (0x1.b0f0b7a76578fp-7 + T * (0x1.112d3541e72fap-19 + T * (-0x1.79921013a4d49p-28 + T * 0x1.0bd243305f727p-39)))) + -0x1.b43428f5c28f6p+13)), f[34], tmp);
      tmp = fma(-(0x1.81f10d173fb7ap+7 * (T * (0x1.0d327faf0cc86p+0 + T * (0x1.a9da4403baf59p-7 + T * (0x1.a9ed607f586a5p-21 + T * (-0x1.50e3cbe90afe8p-28 + T * 0x1.07d55cdad8895p-39)))) + 0x1.4c3ee76c8b439p+13)), f[35], tmp);
    }
    f[36] = tmp / cpm;
  }
};

}  // namespace tgr
