/* Generated by tiger_nga_amd/mech/lanegen.py from the compiled mechanism ethyred
 * (reference combustion/EthyRedF.f90).  Do not edit.  Lane-per-state right-hand side of
 * finitechem_compute_rhs (combustion/finitechem.f90:93-175). */
#pragma once
#include "lane_rhs.h"

namespace tgr {

template <>
struct LaneRhs<46> {
  // production rates cd (kmol/m3/s) from the concentrations, temperature and pressure of this lane's state
  static __device__ __forceinline__ void rates(const double (&C)[45], double T, double P, double (&cd)[45]) {
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
    const double C36 = C[36];
    const double C37 = C[37];
    const double C38 = C[38];
    const double C39 = C[39];
    const double C40 = C[40];
    const double C41 = C[41];
    const double C42 = C[42];
    const double C43 = C[43];
    const double C44 = C[44];
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
    ctot += C36;
    ctot += C37;
    ctot += C38;
    ctot += C39;
    ctot += C40;
    ctot += C41;
    ctot += C42;
    ctot += C43;
    ctot += C44;
    auto M0 = [&]() { double s_ = ctot; s_ = fma(-0x1.0000000000000p+0, C2, s_); s_ = fma(-0x1.0000000000000p+0, C5, s_); s_ = fma(-0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+0, C20, s_); s_ = fma(0x1.0000000000000p+1, C29, s_); return s_; };
    auto M1 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C2, s_); s_ = fma(0x1.6000000000000p+3, C5, s_); s_ = fma(0x1.8000000000000p-1, C10, s_); s_ = fma(0x1.4ccccc0000000p+1, C16, s_); s_ = fma(0x1.0000000000000p+0, C20, s_); s_ = fma(0x1.0000000000000p+1, C29, s_); return s_; };
    auto M2 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C2, s_); s_ = fma(0x1.5333340000000p+2, C5, s_); s_ = fma(0x1.8000000000000p-1, C10, s_); s_ = fma(0x1.4ccccc0000000p+1, C16, s_); s_ = fma(0x1.0000000000000p+0, C20, s_); s_ = fma(0x1.0000000000000p+1, C29, s_); return s_; };
    auto M3 = [&]() { double s_ = ctot; s_ = fma(-0x1.0000000000000p-2, C2, s_); s_ = fma(0x1.5c7ae20000000p+3, C5, s_); s_ = fma(-0x1.3333300000000p-3, C7, s_); s_ = fma(0x1.70a3e00000000p-4, C10, s_); s_ = fma(0x1.2e147c0000000p+0, C16, s_); return s_; };
    auto M4 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C2, s_); s_ = fma(0x1.4000000000000p+2, C5, s_); s_ = fma(0x1.0000000000000p-1, C10, s_); s_ = fma(0x1.0000000000000p+0, C16, s_); s_ = fma(0x1.0000000000000p+1, C20, s_); s_ = fma(0x1.0000000000000p+1, C29, s_); return s_; };
    auto M5 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C2, s_); s_ = fma(0x1.6000000000000p+3, C5, s_); s_ = fma(0x1.8000000000000p-1, C10, s_); s_ = fma(0x1.4ccccc0000000p+1, C16, s_); s_ = fma(0x1.0000000000000p+0, C20, s_); s_ = fma(0x1.0000000000000p+1, C29, s_); return s_; };
    auto M6 = [&]() { double s_ = ctot; s_ = fma(0x1.0000000000000p+0, C2, s_); s_ = fma(-0x1.0000000000000p+0, C5, s_); s_ = fma(0x1.8000000000000p-1, C10, s_); s_ = fma(0x1.4ccccc0000000p+1, C16, s_); s_ = fma(0x1.0000000000000p+0, C20, s_); s_ = fma(0x1.0000000000000p+1, C29, s_); return s_; };
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
    double cd36 = 0.0;
    double cd37 = 0.0;
    double cd38 = 0.0;
    double cd39 = 0.0;
    double cd40 = 0.0;
    double cd41 = 0.0;
    double cd42 = 0.0;
    double cd43 = 0.0;
    double cd44 = 0.0;
    {  // R2 (elementary)
    const double kf = 0x1.c4138c8783e65p+29 * fexp2(fma(-0x1.8fa0b00000000p+24, irt, 0x1.59999a0000000p+1 * lt));
    const double kb = 0x1.b09beee7aedabp+28 * fexp2(fma(-0x1.32b5e60000000p+24, irt, 0x1.54f90a0000000p+1 * lt));
    const double q = kf * C3 * C2 - kb * C4 * C1;
    cd1 += q;
    cd2 -= q;
    cd3 -= q;
    cd4 += q;
    }
    {  // R3 (elementary)
    const double kf = 0x1.fc9bd5fddb67fp+30 * fexp2(fma(-0x1.b5ed600000000p+23, irt, 0x1.828f5c0000000p+0 * lt));
    const double kb = 0x1.6e268e0975208p+33 * fexp2(fma(-0x1.273c980000000p+26, irt, 0x1.6800000000000p+0 * lt));
    const double q = kf * C4 * C2 - kb * C5 * C1;
    cd1 += q;
    cd2 -= q;
    cd4 -= q;
    cd5 += q;
    }
    {  // R4 (elementary)
    const double kf = 0x1.e1645174bab52p+26 * fexp2(fma(0x1.0d78600000000p+23, irt, 0x1.3333340000000p+1 * lt));
    const double kb = 0x1.6a2cb0cfb1368p+30 * fexp2(fma(-0x1.cc15240000000p+25, irt, 0x1.2a8c6a0000000p+1 * lt));
    const double q = kf * C4 * C4 - kb * C5 * C3;
    cd3 += q;
    cd4 = fma(-0x1.0000000000000p+1, q, cd4);
    cd5 += q;
    }
    {  // R1 (elementary)
    const double kf = 0x1.7843b02d8edbcp+38 * fexp2(fma(-0x1.0ffce80000000p+26, irt, -0x1.570a3e0000000p-1 * lt));
    const double kb = 0x1.6ca1517eac207p+33 * fexp2(fma(-0x1.d45d120000000p+18, irt, -0x1.dfd3f60000000p-3 * lt));
    const double q = kf * C1 * C7 - kb * C4 * C3;
    cd1 -= q;
    cd3 += q;
    cd4 += q;
    cd7 -= q;
    }
    {  // R19 (elementary)
    const double kf = 0x1.2309ce5400000p+43 * fexp2(fma(-0x1.149a8c0000000p+26, irt, 0.0 * lt));
    const double kb = 0x1.4561d91d0b10ap+46 * fexp2(fma(-0x1.5b1dde0000000p+28, irt, 0x1.0886e00000000p-2 * lt));
    const double q = kf * C8 * C4 - kb * C7 * C5;
    cd4 -= q;
    cd5 += q;
    cd7 += q;
    cd8 -= q;
    }
    {  // R18 (elementary)
    const double kf = 0x1.62a5cb8000000p+34 * fexp2(fma(0x1.fe41000000000p+20, irt, 0.0 * lt));
    const double kb = 0x1.8c7f6cffb4e41p+37 * fexp2(fma(-0x1.13f8fa0000000p+28, irt, 0x1.0886e00000000p-2 * lt));
    const double q = kf * C8 * C4 - kb * C7 * C5;
    cd4 -= q;
    cd5 += q;
    cd7 += q;
    cd8 -= q;
    }
    {  // R16 (elementary)
    const double kf = 0x1.170634d000000p+36 * fexp2(fma(-0x1.44b5000000000p+21, irt, 0.0 * lt));
    const double q = kf * C8 * C1;
    cd1 -= q;
    cd4 = fma(0x1.0000000000000p+1, q, cd4);
    cd8 -= q;
    }
    {  // R17 (elementary)
    const double kf = 0x1.2a05f20000000p+35 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C8 * C3;
    cd3 -= q;
    cd4 += q;
    cd7 += q;
    cd8 -= q;
    }
    {  // R15 (elementary)
    const double kf = 0x1.d942c90000000p+31 * fexp2(fma(-0x1.5704800000000p+21, irt, 0.0 * lt));
    const double q = kf * C8 * C1;
    cd1 -= q;
    cd3 += q;
    cd5 += q;
    cd8 -= q;
    }
    {  // R13 (elementary)
    const double kf = 0x1.5c90c73ffca62p+30 * fexp2(fma(0x1.172cc00000000p+22, irt, 0x1.08b43a0000000p+1 * lt));
    const double q = kf * C1 * C8;
    cd1 -= q;
    cd2 += q;
    cd7 += q;
    cd8 -= q;
    }
    {  // R26 (elementary)
    const double kf = 0x1.91bca8b63554cp+64 * fexp2(fma(-0x1.2c10680000000p+27, irt, -0x1.c000000000000p+2 * lt));
    const double q = kf * C6 * C4;
    cd4 -= q;
    cd5 += q;
    cd6 -= q;
    cd8 += q;
    }
    {  // RG04 (elementary)
    const double kf = 0x1.a8aedf4000000p+35 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C9 * C3;
    cd1 += q;
    cd3 -= q;
    cd9 -= q;
    cd10 += q;
    }
    {  // RG05 (elementary)
    const double kf = 0x1.bf08eb0000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C9 * C4;
    cd1 += q;
    cd4 -= q;
    cd9 -= q;
    cd11 += q;
    }
    {  // RG09 (elementary)
    const double kf = 0x1.f3ef17e000000p+35 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C9 * C7;
    cd3 += q;
    cd7 -= q;
    cd9 -= q;
    cd11 += q;
    }
    {  // RG06 (elementary)
    const double kf = 0x1.9254d38000000p+36 * fexp2(fma(-0x1.8d08a00000000p+23, irt, 0.0 * lt));
    const double kb = 0x1.081cab6f1a326p+38 * fexp2(fma(-0x1.9cd9300000000p+20, irt, -0x1.2b7cbc0000000p-2 * lt));
    const double q = kf * C9 * C2 - kb * C1 * C12;
    cd1 += q;
    cd2 -= q;
    cd9 -= q;
    cd12 += q;
    }
    {  // RG08 (elementary)
    const double kf = 0x1.5457af8000000p+32 * fexp2(fma(0x1.81be000000000p+21, irt, 0.0 * lt));
    const double q = kf * C9 * C5;
    cd1 += q;
    cd5 -= q;
    cd9 -= q;
    cd14 += q;
    }
    {  // RG38 (elementary)
    const double kf = 0x1.bf08eb0000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.b9fb5ac9f9a01p+33 * fexp2(fma(-0x1.1c99660000000p+25, irt, -0x1.fe3fd60000000p-5 * lt));
    const double q = kf * C15 * C5 - kb * C5 * C12;
    cd12 += q;
    cd15 -= q;
    }
    {  // RG39 (elementary)
    const double kf = 0x1.35630d4f905a4p+28 * fexp2(fma(0x1.dd4b800000000p+21, irt, 0x1.0000000000000p-2 * lt));
    const double q = kf * C15 * C5;
    cd2 += q;
    cd5 -= q;
    cd14 += q;
    cd15 -= q;
    }
    {  // RG35 (elementary)
    const double kf = 0x1.a13b860000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C15 * C7;
    cd1 += q;
    cd4 += q;
    cd7 -= q;
    cd10 += q;
    cd15 -= q;
    }
    {  // RG34 (elementary)
    const double kf = 0x1.04c533c000000p+36 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.1452c52ef394ap+39 * fexp2(fma(-0x1.0528200000000p+26, irt, -0x1.264abe0000000p-1 * lt));
    const double q = kf * C15 * C2 - kb * C1 * C13;
    cd1 += q;
    cd2 -= q;
    cd13 += q;
    cd15 -= q;
    }
    {  // RG31 (elementary)
    const double kf = 0x1.bf08eb0000000p+33 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C15 * C3;
    cd2 += q;
    cd3 -= q;
    cd10 += q;
    cd15 -= q;
    }
    {  // RG36 (elementary)
    const double kf = 0x1.65a0bc0000000p+33 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C15 * C7;
    cd5 += q;
    cd7 -= q;
    cd10 += q;
    cd15 -= q;
    }
    {  // RG30 (elementary)
    const double kf = 0x1.bf08eb0000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.50a4e34f56fe2p+32 * fexp2(fma(-0x1.72f4c40000000p+25, irt, 0x1.d769aa0000000p-3 * lt));
    const double q = kf * C15 * C1 - kb * C2 * C9;
    cd1 -= q;
    cd2 += q;
    cd9 += q;
    cd15 -= q;
    }
    {  // RG33 (elementary)
    const double kf = 0x1.bf08eb0000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C15 * C4;
    cd1 += q;
    cd4 -= q;
    cd14 += q;
    cd15 -= q;
    }
    {  // RG19 (elementary)
    const double kf = 0x1.59b4fa0000000p+32 * fexp2(fma(-0x1.7f4d000000000p+22, irt, 0.0 * lt));
    const double q = kf * C12 * C7;
    cd1 = fma(0x1.0000000000000p+1, q, cd1);
    cd7 -= q;
    cd12 -= q;
    cd16 += q;
    }
    {  // RG17 (elementary)
    const double kf = 0x1.6120000000000p+31 * fexp2(fma(-0x1.7efee00000000p+23, irt, 0x1.0000000000000p+1 * lt));
    const double kb = 0x1.834336177dcd5p+32 * fexp2(fma(-0x1.4b8c760000000p+26, irt, 0x1.1827fa0000000p+1 * lt));
    const double q = kf * C12 * C4 - kb * C5 * C9;
    cd4 -= q;
    cd5 += q;
    cd9 += q;
    cd12 -= q;
    }
    {  // RG20 (elementary)
    const double kf = 0x1.1e1a300000000p+31 * fexp2(fma(-0x1.7f4d000000000p+22, irt, 0.0 * lt));
    const double q = kf * C12 * C7;
    cd3 += q;
    cd7 -= q;
    cd12 -= q;
    cd14 += q;
    }
    {  // RG16 (elementary)
    const double kf = 0x1.2a05f20000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C12 * C4;
    cd1 += q;
    cd4 -= q;
    cd12 -= q;
    cd14 += q;
    }
    {  // RG25 (elementary)
    const double kf = 0x1.2a05f20000000p+35 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C12 * C9;
    cd1 += q;
    cd9 -= q;
    cd12 -= q;
    cd17 += q;
    }
    {  // RG21 (elementary)
    const double kf = 0x1.2a05f20000000p+32 * fexp2(fma(-0x1.7f4d000000000p+22, irt, 0.0 * lt));
    const double q = kf * C12 * C7;
    cd1 += q;
    cd4 += q;
    cd7 -= q;
    cd10 += q;
    cd12 -= q;
    }
    {  // RG18 (elementary)
    const double kf = 0x1.f400000000000p+26 * fexp2(fma(-0x1.cd94100000000p+24, irt, 0x1.0000000000000p+1 * lt));
    const double kb = 0x1.0bf1932336de1p+31 * fexp2(fma(-0x1.d480e20000000p+25, irt, 0x1.7ccccc0000000p+0 * lt));
    const double q = kf * C12 * C2 - kb * C13 * C1;
    cd1 += q;
    cd2 -= q;
    cd12 -= q;
    cd13 += q;
    }
    {  // RG26 (elementary)
    const double kf = 0x1.74876e8000000p+40 * fexp2(fma(-0x1.7d3da80000000p+25, irt, 0.0 * lt));
    const double q = kf * C12 * C12;
    cd2 += q;
    cd12 = fma(-0x1.0000000000000p+1, q, cd12);
    cd17 += q;
    }
    {  // RG15 (elementary)
    const double kf = 0x1.2a05f20000000p+36 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C12 * C3;
    cd1 += q;
    cd3 -= q;
    cd11 += q;
    cd12 -= q;
    }
    {  // RG69 (elementary)
    const double kf = 0x1.bf08eb0000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C13 * C9;
    cd1 += q;
    cd9 -= q;
    cd13 -= q;
    cd18 += q;
    }
    {  // RG52 (elementary)
    const double kf = 0x1.78ffd74000000p+35 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C13 * C3;
    cd1 += q;
    cd3 -= q;
    cd13 -= q;
    cd14 += q;
    }
    {  // RG55 (elementary)
    const double kf = 0x1.20a47438ebc8ep+30 * fexp2(fma(-0x1.5a11c00000000p+24, irt, 0x1.99999a0000000p+0 * lt));
    const double kb = 0x1.83c898230db90p+28 * fexp2(fma(-0x1.a04fdc0000000p+25, irt, 0x1.011f0c0000000p+1 * lt));
    const double q = kf * C13 * C4 - kb * C5 * C12;
    cd4 -= q;
    cd5 += q;
    cd12 += q;
    cd13 -= q;
    }
    {  // RG72 (elementary)
    const double kf = 0x1.74876e8000000p+36 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C13 * C12;
    cd1 += q;
    cd12 -= q;
    cd13 -= q;
    cd19 += q;
    }
    {  // RG74 (elementary)
    const double kf = 0x1.7c64c3796fee8p+33 * fexp2(fma(-0x1.525d180000000p+25, irt, 0x1.99999a0000000p-4 * lt));
    const double kb = 0x1.2ce37effcfaafp+40 * fexp2(fma(-0x1.b754800000000p+22, irt, -0x1.1717580000000p+0 * lt));
    const double q = kf * C13 * C13 - kb * C1 * C21;
    cd1 += q;
    cd13 = fma(-0x1.0000000000000p+1, q, cd13);
    cd21 += q;
    }
    {  // RG53 (elementary)
    const double kf = 0x1.f62b4c4000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C13 * C3;
    cd1 += q;
    cd2 += q;
    cd3 -= q;
    cd10 += q;
    cd13 -= q;
    }
    {  // RG59 (elementary)
    const double kf = 0x1.17e7460000000p+29 * fexp2(fma(-0x1.b9d1780000000p+25, irt, 0.0 * lt));
    const double q = kf * C13 * C7;
    cd4 += q;
    cd7 -= q;
    cd13 -= q;
    cd14 += q;
    }
    {  // RG57 (elementary)
    const double kf = 0x1.18ed6c6cf0030p+37 * fexp2(fma(-0x1.69f0400000000p+22, irt, -0x1.570a3e0000000p+0 * lt));
    const double kb = 0x1.7db9d8730f91dp+36 * fexp2(fma(-0x1.f5cee60000000p+18, irt, -0x1.bce7ee0000000p-1 * lt));
    const double q = kf * C13 * C4 - kb * C5 * C15;
    cd4 -= q;
    cd5 += q;
    cd13 -= q;
    cd15 += q;
    }
    {  // RG91 (elementary)
    const double kf = 0x1.602c1d5682825p+33 * fexp2(fma(-0x1.1281700000000p+25, irt, 0x1.8000000000000p+0 * lt));
    const double kb = 0x1.29cdb5b54fcfap+26 * fexp2(fma(-0x1.401bf20000000p+24, irt, 0x1.fbeb5c0000000p+0 * lt));
    const double q = kf * C20 * C3 - kb * C4 * C13;
    cd3 -= q;
    cd4 += q;
    cd13 += q;
    cd20 -= q;
    }
    {  // RG93 (elementary)
    const double kf = 0x1.bf08eb0000000p+35 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C20 * C9;
    cd1 += q;
    cd9 -= q;
    cd19 += q;
    cd20 -= q;
    }
    {  // RG92 (elementary)
    const double kf = 0x1.01b767c51baa3p+31 * fexp2(fma(-0x1.8e41200000000p+23, irt, 0x1.99999a0000000p+0 * lt));
    const double kb = 0x1.47e5d66ad8d5ep+27 * fexp2(fma(-0x1.0048060000000p+26, irt, 0x1.021b5c0000000p+1 * lt));
    const double q = kf * C20 * C4 - kb * C5 * C13;
    cd4 -= q;
    cd5 += q;
    cd13 += q;
    cd20 -= q;
    }
    {  // RG90 (elementary)
    const double kf = 0x1.e1bd1111ffb19p+33 * fexp2(fma(-0x1.5a11c00000000p+25, irt, 0x1.9eb8520000000p+0 * lt));
    const double kb = 0x1.a9b2c04082075p+27 * fexp2(fma(-0x1.1613ae0000000p+25, irt, 0x1.11f2660000000p+1 * lt));
    const double q = kf * C20 * C1 - kb * C2 * C13;
    cd1 -= q;
    cd2 += q;
    cd13 += q;
    cd20 -= q;
    }
    {  // R28 (elementary)
    const double kf = 0x1.c8cd47ba0ed45p+30 * fexp2(fma(-0x1.d55c400000000p+24, irt, 0x1.1eb8520000000p-3 * lt));
    const double kb = 0x1.a689f8bb1d371p+41 * fexp2(fma(-0x1.0818500000000p+27, irt, -0x1.232e9c0000000p+0 * lt));
    const double q = kf * C10 * C4 - kb * C1 * C16;
    cd1 += q;
    cd4 -= q;
    cd10 -= q;
    cd16 += q;
    }
    {  // R31 (elementary)
    const double kf = 0x1.c086634000000p+34 * fexp2(fma(-0x1.6f169c0000000p+26, irt, 0.0 * lt));
    const double q = kf * C10 * C8;
    cd4 += q;
    cd8 -= q;
    cd10 -= q;
    cd16 += q;
    }
    {  // R29 (elementary)
    const double kf = 0x1.93dc99b504357p+26 * fexp2(fma(0x1.1170000000000p+16, irt, 0x1.eb851e0000000p-6 * lt));
    const double kb = 0x1.7591d14fee88ap+37 * fexp2(fma(-0x1.9a95320000000p+26, irt, -0x1.3f57920000000p+0 * lt));
    const double q = kf * C10 * C4 - kb * C1 * C16;
    cd1 += q;
    cd4 -= q;
    cd10 -= q;
    cd16 += q;
    }
    {  // RG40 (elementary)
    const double kf = 0x1.0c388d0000000p+33 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.093069ac5137bp+32 * fexp2(fma(-0x1.1c99660000000p+25, irt, -0x1.fe3fd60000000p-5 * lt));
    const double q = kf * C15 * C10 - kb * C10 * C12;
    cd12 += q;
    cd15 -= q;
    }
    {  // R32 (elementary)
    const double kf = 0x1.bf08eb0000000p+36 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C11 * C1;
    cd1 -= q;
    cd2 += q;
    cd10 += q;
    cd11 -= q;
    }
    {  // R37 (elementary)
    const double kf = 0x1.fd51291300000p+41 * fexp2(fma(-0x1.0f56e40000000p+26, irt, -0x1.0000000000000p+0 * lt));
    const double kb = 0x1.a483b8abd4cbfp+31 * fexp2(fma(-0x1.46ee300000000p+22, irt, -0x1.88d9fa0000000p-1 * lt));
    const double q = kf * C11 * C5 - kb * C5 * C1 * C10;
    cd1 += q;
    cd10 += q;
    cd11 -= q;
    }
    {  // R38 (elementary)
    const double kf = 0x1.bfbe8719ddf58p+30 * fexp2(fma(0x1.7318000000000p+21, irt, 0x1.9eb8520000000p-1 * lt));
    const double q = kf * C11 * C7;
    cd7 -= q;
    cd8 += q;
    cd10 += q;
    cd11 -= q;
    }
    {  // R33 (elementary)
    const double kf = 0x1.bf08eb0000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C11 * C3;
    cd3 -= q;
    cd4 += q;
    cd10 += q;
    cd11 -= q;
    }
    {  // R35 (elementary)
    const double kf = 0x1.c203db8000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C11 * C4;
    cd4 -= q;
    cd5 += q;
    cd10 += q;
    cd11 -= q;
    }
    {  // R34 (elementary)
    const double kf = 0x1.bf08eb0000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C11 * C3;
    cd1 += q;
    cd3 -= q;
    cd11 -= q;
    cd16 += q;
    }
    {  // RG70 (elementary)
    const double kf = 0x1.8ae17a4000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C13 * C11;
    cd10 += q;
    cd11 -= q;
    cd13 -= q;
    cd20 += q;
    }
    {  // RG46 (elementary)
    const double kf = 0x1.229298c000000p+35 * fexp2(fma(-0x1.c3f7200000000p+23, irt, 0.0 * lt));
    const double q = kf * C14 * C3;
    cd3 -= q;
    cd4 += q;
    cd11 += q;
    cd14 -= q;
    }
    {  // RG71 (elementary)
    const double kf = 0x1.03c958f262512p+27 * fexp2(fma(-0x1.7625400000000p+24, irt, 0x1.67ae140000000p+1 * lt));
    const double q = kf * C13 * C14;
    cd11 += q;
    cd13 -= q;
    cd14 -= q;
    cd20 += q;
    }
    {  // RG47 (elementary)
    const double kf = 0x1.41bee09672314p+32 * fexp2(fma(0x1.c88b000000000p+20, irt, 0x1.2e147a0000000p+0 * lt));
    const double q = kf * C14 * C4;
    cd4 -= q;
    cd5 += q;
    cd11 += q;
    cd14 -= q;
    }
    {  // RG50 (elementary)
    const double kf = 0x1.6069972000000p+36 * fexp2(fma(0x1.07ac000000000p+21, irt, 0.0 * lt));
    const double q = kf * C14 * C9;
    cd1 += q;
    cd9 -= q;
    cd14 -= q;
    cd22 += q;
    }
    {  // RG45 (elementary)
    const double kf = 0x1.e09f93403f5d2p+32 * fexp2(fma(-0x1.5e09600000000p+23, irt, 0x1.e666660000000p+0 * lt));
    const double kb = 0x1.a6ce6c32cbb98p+27 * fexp2(fma(-0x1.1def4c0000000p+26, irt, 0x1.2cbac80000000p+1 * lt));
    const double q = kf * C14 * C1 - kb * C2 * C11;
    cd1 -= q;
    cd2 += q;
    cd11 += q;
    cd14 -= q;
    }
    {  // RG89 (elementary)
    const double kf = 0x1.0c388d0000000p+34 * fexp2(fma(-0x1.cc34800000000p+21, irt, 0.0 * lt));
    const double q = kf * C24 * C7;
    cd7 -= q;
    cd8 += q;
    cd14 += q;
    cd24 -= q;
    }
    {  // RG86 (elementary)
    const double kf = 0x1.16c75b7ab6bb9p+34 * fexp2(fma(-0x1.3747800000000p+21, irt, -0x1.70a3d80000000p-4 * lt));
    const double kb = 0x1.0f48debe4b33ap+29 * fexp2(fma(-0x1.81d7d80000000p+23, irt, 0x1.5beea20000000p+0 * lt));
    const double q = kf * C24 * C1 - kb * C5 * C15;
    cd1 -= q;
    cd5 += q;
    cd15 += q;
    cd24 -= q;
    }
    {  // RG85 (elementary)
    const double kf = 0x1.1ba28006d2a53p+33 * fexp2(fma(0x1.2287000000000p+20, irt, 0x1.4ccccc0000000p-1 * lt));
    const double kb = 0x1.9642fa000f416p+28 * fexp2(fma(-0x1.b4fec00000000p+23, irt, 0x1.a0c9320000000p+0 * lt));
    const double q = kf * C24 * C1 - kb * C4 * C13;
    cd1 -= q;
    cd4 += q;
    cd13 += q;
    cd24 -= q;
    }
    {  // RG84 (elementary)
    const double kf = 0x1.2a05f20000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C24 * C1;
    cd1 -= q;
    cd2 += q;
    cd14 += q;
    cd24 -= q;
    }
    {  // RG41 (elementary)
    const double kf = 0x1.a13b860000000p+32 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.9c84329a494e9p+31 * fexp2(fma(-0x1.1c99660000000p+25, irt, -0x1.fe3fd60000000p-5 * lt));
    const double q = kf * C15 * C16 - kb * C16 * C12;
    cd12 += q;
    cd15 -= q;
    }
    {  // RG42 (elementary)
    const double kf = 0x1.a13b860000000p+33 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C15 * C16;
    cd10 += q;
    cd14 += q;
    cd15 -= q;
    cd16 -= q;
    }
    {  // RG11 (elementary)
    const double kf = 0x1.61e70f6000000p+37 * fexp2(fma(-0x1.f812f80000000p+25, irt, 0.0 * lt));
    const double q = kf * C9 * C16;
    cd9 -= q;
    cd10 += q;
    cd11 += q;
    cd16 -= q;
    }
    {  // RG108 (elementary)
    const double kf = 0x1.05da7719381d3p+32 * fexp2(fma(-0x1.cc34800000000p+21, irt, 0x1.2147ae0000000p+1 * lt));
    const double kb = 0x1.21634bb1b3e6cp+38 * fexp2(fma(-0x1.e515080000000p+26, irt, 0x1.a9d8840000000p+0 * lt));
    const double q = kf * C25 * C2 - kb * C1 * C17;
    cd1 += q;
    cd2 -= q;
    cd17 += q;
    cd25 -= q;
    }
    {  // RG107 (elementary)
    const double kf = 0x1.2a05f20000000p+33 * fexp2(fma(0x1.81be000000000p+21, irt, 0.0 * lt));
    const double q = kf * C25 * C7;
    cd7 -= q;
    cd10 += q;
    cd11 += q;
    cd25 -= q;
    }
    {  // RG105 (elementary)
    const double kf = 0x1.74876e8000000p+35 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C25 * C3;
    cd3 -= q;
    cd9 += q;
    cd10 += q;
    cd25 -= q;
    }
    {  // RG106 (elementary)
    const double kf = 0x1.2a05f20000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C25 * C4;
    cd1 += q;
    cd4 -= q;
    cd23 += q;
    cd25 -= q;
    }
    {  // RR017 (elementary)
    const double kf = 0x1.671e344000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.4770b14b43a48p+42 * fexp2(fma(-0x1.3126616000000p+27, irt, -0x1.60bcbe0000000p+0 * lt));
    const double q = kf * C25 * C13 - kb * C1 * C26;
    cd1 += q;
    cd13 -= q;
    cd25 -= q;
    cd26 += q;
    }
    {  // RG118 (elementary)
    const double kf = 0x1.0db6054000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.377d9c87e8238p+41 * fexp2(fma(-0x1.edee180000000p+26, irt, -0x1.1eeb0c0000000p-1 * lt));
    const double q = kf * C25 * C4 - kb * C3 * C17;
    cd3 += q;
    cd4 -= q;
    cd17 += q;
    cd25 -= q;
    }
    {  // RG121 (elementary)
    const double kf = 0x1.c697f96b20fcdp+26 * fexp2(fma(-0x1.0cdc200000000p+23, irt, 0x1.8ccccc0000000p+0 * lt));
    const double q = kf * C17 * C4;
    cd1 += q;
    cd4 -= q;
    cd17 -= q;
    cd22 += q;
    }
    {  // RG117 (elementary)
    const double kf = 0x1.86a0000000000p+31 * fexp2(fma(-0x1.e53ac00000000p+22, irt, 0x1.0000000000000p+1 * lt));
    const double q = kf * C17 * C3;
    cd3 -= q;
    cd10 += q;
    cd12 += q;
    cd17 -= q;
    }
    {  // RR008 (elementary)
    const double kf = 0x1.229298c000000p+36 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.e2e0049c2accap+53 * fexp2(fma(-0x1.de56460000000p+27, irt, -0x1.4caea80000000p+0 * lt));
    const double q = kf * C17 * C25 - kb * C27;
    cd17 -= q;
    cd25 -= q;
    cd27 += q;
    }
    {  // RG119 (elementary)
    const double kf = 0x1.89abdfad03212p+30 * fexp2(fma(-0x1.104b080000000p+26, irt, 0x1.11eb860000000p+1 * lt));
    const double kb = 0x1.0070ec55f581ep+27 * fexp2(fma(-0x1.50b4740000000p+23, irt, 0x1.50ff440000000p+1 * lt));
    const double q = kf * C17 * C4 - kb * C5 * C25;
    cd4 -= q;
    cd5 += q;
    cd17 -= q;
    cd25 += q;
    }
    {  // RG116 (elementary)
    const double kf = 0x1.fa40000000000p+30 * fexp2(fma(-0x1.e53ac00000000p+22, irt, 0x1.0000000000000p+1 * lt));
    const double q = kf * C17 * C3;
    cd1 += q;
    cd3 -= q;
    cd17 -= q;
    cd23 += q;
    }
    {  // RR004 (elementary)
    const double kf = 0x1.61e70f6000000p+37 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.3565141dcb299p+42 * fexp2(fma(-0x1.90c17e0000000p+26, irt, -0x1.5b2b560000000p+0 * lt));
    const double q = kf * C17 * C15 - kb * C1 * C26;
    cd1 += q;
    cd15 -= q;
    cd17 -= q;
    cd26 += q;
    }
    {  // RG122 (elementary)
    const double kf = 0x1.cfe9e65812dcap+26 * fexp2(fma(-0x1.4948e00000000p+23, irt, 0x1.75c2900000000p-1 * lt));
    const double q = kf * C17 * C4;
    cd4 -= q;
    cd10 += q;
    cd13 += q;
    cd17 -= q;
    }
    {  // RG130 (elementary)
    const double kf = 0x1.bf08eb0000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.66a4b3919dba1p+36 * fexp2(fma(-0x1.110714a000000p+28, irt, 0x1.6d43d00000000p-3 * lt));
    const double q = kf * C18 * C1 - kb * C2 * C17;
    cd1 -= q;
    cd2 += q;
    cd17 += q;
    cd18 -= q;
    }
    {  // RB07 (elementary)
    const double kf = 0x1.c9c3800000000p+29 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C18 * C18;
    cd17 += q;
    cd18 = fma(-0x1.0000000000000p+1, q, cd18);
    cd19 += q;
    }
    {  // RR011 (elementary)
    const double kf = 0x1.4f46b04000000p+36 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C18 * C11;
    cd10 += q;
    cd11 -= q;
    cd18 -= q;
    cd19 += q;
    }
    {  // RR013 (elementary)
    const double kf = 0x1.0d1d6ec000000p+33 * fexp2(fma(0x1.86a0000000000p+21, irt, 0.0 * lt));
    const double q = kf * C18 * C13;
    cd13 -= q;
    cd17 += q;
    cd18 -= q;
    cd20 += q;
    }
    {  // RG132 (elementary)
    const double kf = 0x1.2a05f20000000p+32 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C18 * C4;
    cd4 -= q;
    cd5 += q;
    cd17 += q;
    cd18 -= q;
    }
    {  // RG133 (elementary)
    const double kf = 0x1.d67d340aeeacdp+24 * fexp2(fma(0x1.8911000000000p+20, irt, 0x1.9c28f60000000p+0 * lt));
    const double q = kf * C18 * C7;
    cd7 -= q;
    cd8 += q;
    cd17 += q;
    cd18 -= q;
    }
    {  // RG135 (elementary)
    const double kf = 0x1.d4040197c6493p+32 * fexp2(fma(-0x1.0366400000000p+22, irt, -0x1.63d70a0000000p+0 * lt));
    const double q = kf * C18 * C7;
    cd7 -= q;
    cd11 += q;
    cd14 += q;
    cd18 -= q;
    }
    {  // RG159 (elementary)
    const double kf = 0x1.c0a38bec3b72bp+30 * fexp2(fma(-0x1.c4e1800000000p+21, irt, 0x1.5c28f60000000p+0 * lt));
    const double q = kf * C19 * C3;
    cd3 -= q;
    cd11 += q;
    cd13 += q;
    cd19 -= q;
    }
    {  // RIC67 (elementary)
    const double kf = 0x1.8701a80000000p+28 * fexp2(fma(-0x1.cbe6600000000p+24, irt, 0.0 * lt));
    const double q = kf * C19 * C13;
    cd13 -= q;
    cd19 -= q;
    cd28 += q;
    }
    {  // RG162 (elementary)
    const double kf = 0x1.c600000000000p+25 * fexp2(fma(-0x1.25a7c80000000p+25, irt, 0x1.0000000000000p+1 * lt));
    const double kb = 0x1.1e794f5f462b7p+25 * fexp2(fma(-0x1.aa74f60000000p+23, irt, 0x1.f7357e0000000p+0 * lt));
    const double q = kf * C19 * C13 - kb * C20 * C18;
    cd13 -= q;
    cd18 += q;
    cd19 -= q;
    cd20 += q;
    }
    {  // RG160 (elementary)
    const double kf = 0x1.de53a6fde9767p+24 * fexp2(fma(0x1.b774000000000p+21, irt, 0x1.0ccccc0000000p+2 * lt));
    const double kb = 0x1.800473c6e7460p+20 * fexp2(fma(-0x1.8cfbf40000000p+24, irt, 0x1.2541740000000p+2 * lt));
    const double q = kf * C19 * C4 - kb * C5 * C18;
    cd4 -= q;
    cd5 += q;
    cd18 += q;
    cd19 -= q;
    }
    {  // RG158 (elementary)
    const double kf = 0x1.4f6e4c893cde7p+28 * fexp2(fma(-0x1.dada800000000p+21, irt, 0x1.3c28f60000000p+1 * lt));
    const double q = kf * C19 * C3;
    cd3 -= q;
    cd12 += q;
    cd14 += q;
    cd19 -= q;
    }
    {  // RG156 (elementary)
    const double kf = 0x1.ab2ce5a281e06p+31 * fexp2(fma(-0x1.73db500000000p+25, irt, 0x1.6000000000000p+1 * lt));
    const double kb = 0x1.dc61ee0c300c6p+24 * fexp2(fma(-0x1.d34ace0000000p+23, irt, 0x1.9e30fc0000000p+1 * lt));
    const double q = kf * C19 * C1 - kb * C2 * C18;
    cd1 -= q;
    cd2 += q;
    cd18 += q;
    cd19 -= q;
    }
    {  // RG171 (elementary)
    const double kf = 0x1.53dd78d77f5eap+23 * fexp2(fma(0x1.03b4600000000p+23, irt, 0x1.051eb80000000p+0 * lt));
    const double q = kf * C21 * C7;
    cd7 -= q;
    cd8 += q;
    cd19 += q;
    cd21 -= q;
    }
    {  // RR034 (elementary)
    const double kf = 0x1.bf08eb0000000p+36 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C21 * C11;
    cd10 += q;
    cd11 -= q;
    cd21 -= q;
    cd29 += q;
    }
    {  // RG178 (elementary)
    const double kf = 0x1.888d6e5c00000p+39 * fexp2(fma(-0x1.6339800000000p+26, irt, 0.0 * lt));
    const double q = kf * C29 * C13;
    cd13 -= q;
    cd20 += q;
    cd21 += q;
    cd29 -= q;
    }
    {  // RG174 (elementary)
    const double kf = 0x1.a296d773fedecp+31 * fexp2(fma(-0x1.6e84200000000p+24, irt, 0x1.59999a0000000p+1 * lt));
    const double kb = 0x1.49edb290c8afap+24 * fexp2(fma(-0x1.0e5c0e0000000p+25, irt, 0x1.a12cd00000000p+1 * lt));
    const double q = kf * C29 * C1 - kb * C2 * C21;
    cd1 -= q;
    cd2 += q;
    cd21 += q;
    cd29 -= q;
    }
    {  // RG110 (elementary)
    const double kf = 0x1.74876e8000000p+36 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C23 * C3;
    cd1 += q;
    cd3 -= q;
    cd10 = fma(0x1.0000000000000p+1, q, cd10);
    cd23 -= q;
    }
    {  // RG109 (elementary)
    const double kf = 0x1.74876e8000000p+36 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.d3bfa6411ce3ap+30 * fexp2(fma(-0x1.11df060000000p+26, irt, 0x1.8f9f020000000p+0 * lt));
    const double q = kf * C23 * C1 - kb * C10 * C15;
    cd1 -= q;
    cd10 += q;
    cd15 += q;
    cd23 -= q;
    }
    {  // RG114 (elementary)
    const double kf = 0x1.2a05f20000000p+33 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C23 * C23;
    cd10 = fma(0x1.0000000000000p+1, q, cd10);
    cd17 += q;
    cd23 = fma(-0x1.0000000000000p+1, q, cd23);
    }
    {  // RR009 (elementary)
    const double kf = 0x1.7d78400000000p+26 * fexp2(fma(-0x1.7efee00000000p+23, irt, 0.0 * lt));
    const double q = kf * C17 * C23;
    cd10 += q;
    cd17 -= q;
    cd23 -= q;
    cd26 += q;
    }
    {  // RG112 (elementary)
    const double kf = 0x1.74876e8000000p+35 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C23 * C9;
    cd9 -= q;
    cd10 += q;
    cd17 += q;
    cd23 -= q;
    }
    {  // RG113 (elementary)
    const double kf = 0x1.bf08eb0000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C23 * C12;
    cd10 += q;
    cd12 -= q;
    cd18 += q;
    cd23 -= q;
    }
    {  // RR024 (elementary)
    const double kf = 0x1.2a05f20000000p+33 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C23 * C4;
    cd4 -= q;
    cd11 = fma(0x1.0000000000000p+1, q, cd11);
    cd23 -= q;
    }
    {  // RR022 (elementary)
    const double kf = 0x1.74876e8000000p+35 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C23 * C13;
    cd10 += q;
    cd13 -= q;
    cd19 += q;
    cd23 -= q;
    }
    {  // RG124 (elementary)
    const double kf = 0x1.e9f6b45c14e80p+32 * fexp2(fma(-0x1.39b8800000000p+21, irt, 0x1.6147ae0000000p+0 * lt));
    const double kb = 0x1.4bad2a544b696p+25 * fexp2(fma(-0x1.f6fbc00000000p+26, irt, 0x1.7b50b00000000p+1 * lt));
    const double q = kf * C22 * C1 - kb * C10 * C13;
    cd1 -= q;
    cd10 += q;
    cd13 += q;
    cd22 -= q;
    }
    {  // RG123 (elementary)
    const double kf = 0x1.74876e8000000p+35 * fexp2(fma(-0x1.feb6300000000p+24, irt, 0.0 * lt));
    const double kb = 0x1.7b14c1e3a8cb8p+30 * fexp2(fma(-0x1.5751860000000p+24, irt, 0x1.31c0440000000p-1 * lt));
    const double q = kf * C22 * C1 - kb * C2 * C23;
    cd1 -= q;
    cd2 += q;
    cd22 -= q;
    cd23 += q;
    }
    {  // RG127 (elementary)
    const double kf = 0x1.bf08eb0000000p+32 * fexp2(fma(-0x1.fedd400000000p+22, irt, 0.0 * lt));
    const double kb = 0x1.477d53a3fdbdbp+30 * fexp2(fma(-0x1.cd272a0000000p+25, irt, 0x1.f943e20000000p-2 * lt));
    const double q = kf * C22 * C4 - kb * C5 * C23;
    cd4 -= q;
    cd5 += q;
    cd22 -= q;
    cd23 += q;
    }
    {  // RR025 (elementary)
    const double kf = 0x1.2a05f20000000p+32 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C22 * C4;
    cd4 -= q;
    cd10 += q;
    cd22 -= q;
    cd24 += q;
    }
    {  // RR068 (elementary)
    const double kf = 0x1.74876e8000000p+34 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C26 * C11;
    cd10 += q;
    cd11 -= q;
    cd26 -= q;
    cd30 += q;
    }
    {  // RLPP009 (elementary)
    const double kf = 0x1.32d0b8271edb2p+55 * fexp2(fma(-0x1.0d1f820000000p+26, irt, -0x1.3b95820000000p+3 * lt));
    const double kb = 0x1.c4195534635c8p+95 * fexp2(fma(-0x1.42babc0000000p+29, irt, -0x1.6a3afc0000000p+3 * lt));
    const double q = kf * C26 * C26 - kb * C31;
    cd26 = fma(-0x1.0000000000000p+1, q, cd26);
    cd31 += q;
    }
    {  // RR055 (elementary)
    const double kf = 0x1.c3b71e4dfa21bp+43 * fexp2(fma(-0x1.365d200000000p+24, irt, -0x1.43d70a0000000p+2 * lt));
    const double kb = 0x1.4eed875cfb1ccp+60 * fexp2(fma(-0x1.771dfe0000000p+28, irt, -0x1.446a2c0000000p+2 * lt));
    const double q = kf * C26 * C1 - kb * C30;
    cd1 -= q;
    cd26 -= q;
    cd30 += q;
    }
    {  // RR058 (elementary)
    const double kf = 0x1.cfe9e65812dcap+26 * fexp2(fma(-0x1.4948e00000000p+23, irt, 0x1.75c2900000000p-1 * lt));
    const double q = kf * C26 * C4;
    cd4 -= q;
    cd10 += q;
    cd19 += q;
    cd26 -= q;
    }
    {  // RR062 (elementary)
    const double kf = 0x1.a296d773fedecp+22 * fexp2(fma(-0x1.7f4d000000000p+22, irt, 0x1.b333340000000p+0 * lt));
    const double q = kf * C26 * C7;
    cd7 -= q;
    cd11 += q;
    cd22 += q;
    cd26 -= q;
    }
    {  // RP011 (elementary)
    const double kf = 0x1.639a8c6809e91p+52 * fexp2(fma(-0x1.f6da780000000p+26, irt, -0x1.c000000000000p+2 * lt));
    const double kb = 0x1.3d183a513536ep+74 * fexp2(fma(-0x1.f3cac80000000p+27, irt, -0x1.07e0a00000000p+3 * lt));
    const double q = kf * C26 * C26 - kb * C1 * C32;
    cd1 += q;
    cd26 = fma(-0x1.0000000000000p+1, q, cd26);
    cd32 += q;
    }
    {  // RCP16 (elementary)
    const double kf = 0x1.03ad27d4874f5p+63 * fexp2(fma(-0x1.4fb1800000000p+27, irt, -0x1.9000000000000p+3 * lt));
    const double kb = 0x1.e5050747eea43p+92 * fexp2(fma(-0x1.d0fa7c0000000p+28, irt, -0x1.b249ba0000000p+3 * lt));
    const double q = kf * C26 * C17 - kb * C33;
    cd17 -= q;
    cd26 -= q;
    cd33 += q;
    }
    {  // RR089 (elementary)
    const double kf = 0x1.86a0000000000p+30 * fexp2(fma(-0x1.e53ac00000000p+22, irt, 0x1.0000000000000p+1 * lt));
    const double q = kf * C30 * C3;
    cd3 -= q;
    cd10 += q;
    cd19 += q;
    cd30 -= q;
    }
    {  // RR079 (elementary)
    const double kf = 0x1.a9eaabe2b355ep+32 * fexp2(fma(-0x1.6b4fd00000000p+24, irt, 0x1.eb851e0000000p+0 * lt));
    const double q = kf * C30 * C3;
    cd3 -= q;
    cd4 += q;
    cd26 += q;
    cd30 -= q;
    }
    {  // RR080 (elementary)
    const double kf = 0x1.8cf56f9e3ebb4p+29 * fexp2(fma(-0x1.7a6b000000000p+21, irt, 0x1.1c28f60000000p+1 * lt));
    const double kb = 0x1.87099dd162a6ep+26 * fexp2(fma(-0x1.e18e780000000p+26, irt, 0x1.3cdc340000000p+1 * lt));
    const double q = kf * C30 * C4 - kb * C5 * C26;
    cd4 -= q;
    cd5 += q;
    cd26 += q;
    cd30 -= q;
    }
    {  // RR005 (elementary)
    const double kf = 0x1.912f6ea7fbeafp+35 * fexp2(fma(-0x1.5cd0e00000000p+24, irt, 0x1.c28f5c0000000p-2 * lt));
    const double kb = 0x1.4cb08db6dcb85p+28 * fexp2(fma(-0x1.61ae1e0000000p+25, irt, 0x1.949f940000000p+0 * lt));
    const double q = kf * C30 * C1 - kb * C13 * C17;
    cd1 -= q;
    cd13 += q;
    cd17 += q;
    cd30 -= q;
    }
    {  // RR088 (elementary)
    const double kf = 0x1.fa40000000000p+29 * fexp2(fma(-0x1.e53ac00000000p+22, irt, 0x1.0000000000000p+1 * lt));
    const double q = kf * C30 * C3;
    cd3 -= q;
    cd13 += q;
    cd23 += q;
    cd30 -= q;
    }
    {  // RR081 (elementary)
    const double kf = 0x1.8904a3f000000p+38 * fexp2(fma(-0x1.6339800000000p+26, irt, 0.0 * lt));
    const double kb = 0x1.304a78aaabfebp+39 * fexp2(fma(-0x1.353a5ee000000p+27, irt, -0x1.49b5200000000p-3 * lt));
    const double q = kf * C30 * C13 - kb * C20 * C26;
    cd13 -= q;
    cd20 += q;
    cd26 += q;
    cd30 -= q;
    }
    {  // RR078 (elementary)
    const double kf = 0x1.a296d773fedecp+30 * fexp2(fma(-0x1.6e84200000000p+24, irt, 0x1.59999a0000000p+1 * lt));
    const double kb = 0x1.1e636593f9535p+25 * fexp2(fma(-0x1.40dd3c0000000p+26, irt, 0x1.8794860000000p+1 * lt));
    const double q = kf * C30 * C1 - kb * C2 * C26;
    cd1 -= q;
    cd2 += q;
    cd26 += q;
    cd30 -= q;
    }
    {  // RR014 (elementary)
    const double kf = 0x1.6b613d842b8d3p+72 * fexp2(fma(-0x1.be39660000000p+28, irt, -0x1.eae1480000000p+2 * lt));
    const double kb = 0x1.82bc41afccbb5p+47 * fexp2(fma(-0x1.0a6e7c0000000p+25, irt, -0x1.803d9a0000000p+2 * lt));
    const double q = kf * C34 - kb * C13 * C18;
    cd13 += q;
    cd18 += q;
    cd34 -= q;
    }
    {  // RR143 (elementary)
    const double kf = 0x1.68cd914726bb1p+29 * fexp2(fma(0x1.f0d3800000000p+21, irt, 0x1.99999a0000000p+0 * lt));
    const double q = kf * C34 * C3;
    cd3 -= q;
    cd11 += q;
    cd21 += q;
    cd34 -= q;
    }
    {  // RR141 (elementary)
    const double kf = 0x1.37d9656660855p+41 * fexp2(fma(-0x1.64e7300000000p+25, irt, -0x1.31eb860000000p+1 * lt));
    const double kb = 0x1.2def3ee18f50ap+34 * fexp2(fma(-0x1.3266740000000p+26, irt, -0x1.b802e20000000p-1 * lt));
    const double q = kf * C34 * C1 - kb * C13 * C19;
    cd1 -= q;
    cd13 += q;
    cd19 += q;
    cd34 -= q;
    }
    {  // RIC66 (elementary)
    const double kf = 0x1.36d865f0f2725p+34 * fexp2(fma(-0x1.cafc000000000p+22, irt, 0x1.eb851e0000000p-6 * lt));
    const double q = kf * C34 * C1;
    cd1 -= q;
    cd28 += q;
    cd34 -= q;
    }
    {  // RIC64 (elementary)
    const double kf = 0x1.8c74079b8afc4p+21 * fexp2(fma(-0x1.0fcc140000000p+26, irt, 0x1.570a3e0000000p+2 * lt));
    const double q = kf * C28;
    cd13 += q;
    cd19 += q;
    cd28 -= q;
    }
    {  // RIC65 (elementary)
    const double kf = 0x1.ba6718bccb851p+48 * fexp2(fma(-0x1.41ffa40000000p+27, irt, -0x1.970a3e0000000p+0 * lt));
    const double q = kf * C28;
    cd1 += q;
    cd28 -= q;
    cd34 += q;
    }
    {  // RH10 (elementary)
    const double kf = 0x1.28d97f1e72710p+49 * fexp2(fma(-0x1.ecef680000000p+25, irt, -0x1.f7ae140000000p+2 * lt));
    const double kb = 0x1.136136d131b0ep+57 * fexp2(fma(-0x1.7cbcce0000000p+27, irt, -0x1.fb80340000000p+2 * lt));
    const double q = kf * C35 * C1 - kb * C27;
    cd1 -= q;
    cd27 += q;
    cd35 -= q;
    }
    {  // RH07 (elementary)
    const double kf = 0x1.1ce9030000000p+33 * fexp2(fma(-0x1.f05e500000000p+26, irt, 0.0 * lt));
    const double q = kf * C35 * C7;
    cd7 -= q;
    cd23 = fma(0x1.0000000000000p+1, q, cd23);
    cd35 -= q;
    }
    {  // RH12 (elementary)
    const double kf = 0x1.4acd00b4acad1p+29 * fexp2(fma(-0x1.2f58400000000p+23, irt, -0x1.0000000000000p-2 * lt));
    const double q = kf * C35 * C4;
    cd4 -= q;
    cd10 += q;
    cd26 += q;
    cd35 -= q;
    }
    {  // ROX02 (elementary)
    const double kf = 0x1.992a51a049408p+77 * fexp2(fma(-0x1.0f03e20000000p+28, irt, -0x1.34f5c20000000p+4 * lt));
    const double kb = 0x1.048d9fc94d2cbp+104 * fexp2(fma(-0x1.0076ca0000000p+29, irt, -0x1.45930c0000000p+4 * lt));
    const double q = kf * C35 * C17 - kb * C36;
    cd17 -= q;
    cd35 -= q;
    cd36 += q;
    }
    {  // RH17 (elementary)
    const double kf = 0x1.9983b5977f044p+45 * fexp2(fma(-0x1.3f84e00000000p+25, irt, -0x1.ab851e0000000p+1 * lt));
    const double q = kf * C27 * C1;
    cd1 -= q;
    cd17 = fma(0x1.0000000000000p+1, q, cd17);
    cd27 -= q;
    }
    {  // RH19 (elementary)
    const double kf = 0x1.bf08eb0000000p+33 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C27 * C1;
    cd1 -= q;
    cd2 += q;
    cd27 -= q;
    cd35 += q;
    }
    {  // RLPCP18 (elementary)
    const double kf = 0x1.946b853410969p+51 * fexp2(fma(-0x1.8b64b40000000p+26, irt, -0x1.3666660000000p+2 * lt));
    const double q = kf * C33 * C13;
    cd1 = fma(0x1.0000000000000p+1, q, cd1);
    cd13 -= q;
    cd31 += q;
    cd33 -= q;
    }
    {  // RCP17 (elementary)
    const double kf = 0x1.b659fe99df450p+52 * fexp2(fma(-0x1.18f3d40000000p+27, irt, -0x1.01eb860000000p+2 * lt));
    const double q = kf * C33 * C33;
    cd1 = fma(0x1.0000000000000p+1, q, cd1);
    cd33 = fma(-0x1.0000000000000p+1, q, cd33);
    cd37 += q;
    }
    {  // RLPP015 (elementary)
    const double kf = 0x1.73e49d2704e72p+23 * fexp2(fma(-0x1.1d7df00000000p+24, irt, 0x1.1e147a0000000p+2 * lt));
    const double q = kf * C32 * C19;
    cd18 += q;
    cd19 -= q;
    cd31 += q;
    cd32 -= q;
    }
    {  // RI00 (elementary)
    const double kf = 0x1.2a05f20000000p+33 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double kb = 0x1.1ba1e2cfa15ddp+67 * fexp2(fma(-0x1.f1269a0000000p+28, irt, -0x1.0427fa0000000p+1 * lt));
    const double q = kf * C32 * C26 - kb * C38;
    cd26 -= q;
    cd32 -= q;
    cd38 += q;
    }
    {  // RLPOX00 (elementary)
    const double kf = 0x1.8aa79c19f7ce1p+62 * fexp2(fma(-0x1.7fdf7c0000000p+26, irt, -0x1.2cac080000000p+3 * lt));
    const double q = kf * C1 * C32;
    cd1 -= q;
    cd31 += q;
    cd32 -= q;
    }
    {  // RK012 (elementary)
    const double kf = 0x1.18e456752913fp+30 * fexp2(fma(-0x1.93bf600000000p+23, irt, 0x1.0666660000000p+1 * lt));
    const double kb = 0x1.59642f7012e7fp+50 * fexp2(fma(-0x1.6d0a400000000p+27, irt, 0x1.14b1ee0000000p-2 * lt));
    const double q = kf * C32 * C17 - kb * C39;
    cd17 -= q;
    cd32 -= q;
    cd39 += q;
    }
    {  // RLPOX03 (elementary)
    const double kf = 0x1.4c7165f0ac776p+35 * fexp2(fma(-0x1.058e020000000p+26, irt, 0x1.cf9db20000000p+0 * lt));
    const double kb = 0x1.981f3b6e6e9ffp+27 * fexp2(fma(-0x1.86be960000000p+24, irt, 0x1.2fb59e0000000p+1 * lt));
    const double q = kf * C31 * C1 - kb * C2 * C32;
    cd1 -= q;
    cd2 += q;
    cd31 -= q;
    cd32 += q;
    }
    {  // RLPOX04 (elementary)
    const double kf = 0x1.9093b0e50c544p+28 * fexp2(fma(-0x1.8874c00000000p+21, irt, 0x1.5872b00000000p+1 * lt));
    const double q = kf * C31 * C4;
    cd4 -= q;
    cd5 += q;
    cd31 -= q;
    cd32 += q;
    }
    {  // RI03 (elementary)
    const double kf = 0x1.3b93f7d414987p+27 * fexp2(fma(-0x1.6116a00000000p+25, irt, 0x1.3d70a40000000p+1 * lt));
    const double kb = 0x1.fe94c44aeef05p+40 * fexp2(fma(-0x1.8b28fe0000000p+26, irt, 0x1.5c38080000000p+0 * lt));
    const double q = kf * C40 * C17 - kb * C1 * C38;
    cd1 += q;
    cd17 -= q;
    cd38 += q;
    cd40 -= q;
    }
    {  // RT04 (elementary)
    const double kf = 0x1.bcc3ad5e87731p+87 * fexp2(fma(-0x1.10a55d0000000p+28, irt, -0x1.c4cccc0000000p+3 * lt));
    const double kb = 0x1.d0f68db5a8bbfp+76 * fexp2(fma(-0x1.a08e220000000p+27, irt, -0x1.8361e40000000p+3 * lt));
    const double q = kf * C40 * C1 - kb * C13 * C32;
    cd1 -= q;
    cd13 += q;
    cd32 += q;
    cd40 -= q;
    }
    {  // RT20 (elementary)
    const double kf = 0x1.07473e7571cd8p+52 * fexp2(fma(-0x1.7cb4f00000000p+26, irt, -0x1.ef5c280000000p+2 * lt));
    const double q = kf * C40 * C26;
    cd1 = fma(0x1.0000000000000p+1, q, cd1);
    cd26 -= q;
    cd37 += q;
    cd40 -= q;
    }
    {  // RT05 (elementary)
    const double kf = 0x1.74e4905ba0000p+49 * fexp2(fma(-0x1.41e9ab0000000p+28, irt, 0.0 * lt));
    const double kb = 0x1.9331e0e87a48dp+25 * fexp2(fma(-0x1.5fa6480000000p+25, irt, 0x1.1f69440000000p+1 * lt));
    const double q = kf * C40 - kb * C17 * C33;
    cd17 += q;
    cd33 += q;
    cd40 -= q;
    }
    {  // RP106 (elementary)
    const double kf = 0x1.accf5043a82c1p+46 * fexp2(fma(-0x1.7ce5c40000000p+26, irt, -0x1.0f5c280000000p+2 * lt));
    const double kb = 0x1.7c1160b2b7b16p+68 * fexp2(fma(-0x1.5cfe800000000p+28, irt, -0x1.81eda60000000p+2 * lt));
    const double q = kf * C41 * C19 - kb * C1 * C37;
    cd1 += q;
    cd19 -= q;
    cd37 += q;
    cd41 -= q;
    }
    {  // RK100 (elementary)
    const double kf = 0x1.2f35175d75bafp+26 * fexp2(fma(-0x1.47c2400000000p+22, irt, 0x1.4000000000000p+1 * lt));
    const double kb = 0x1.08d33f0c26e04p+57 * fexp2(fma(-0x1.70ac7c0000000p+28, irt, 0x1.f56fb80000000p-1 * lt));
    const double q = kf * C41 * C17 - kb * C42;
    cd17 -= q;
    cd41 -= q;
    cd42 += q;
    }
    {  // RP105 (elementary)
    const double kf = 0x1.509f7984c80a0p+35 * fexp2(fma(-0x1.f701880000000p+25, irt, -0x1.70a3d80000000p+0 * lt));
    const double kb = 0x1.c08c34a501426p+57 * fexp2(fma(-0x1.296bd40000000p+28, irt, -0x1.9148aa0000000p+1 * lt));
    const double q = kf * C43 * C18 - kb * C1 * C37;
    cd1 += q;
    cd18 -= q;
    cd37 += q;
    cd43 -= q;
    }
    {  // RLPST00 (elementary)
    const double kf = 0x1.2a05f20000000p+33 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double q = kf * C43 * C4;
    cd4 -= q;
    cd23 += q;
    cd31 += q;
    cd43 -= q;
    }
    {  // RK017 (elementary)
    const double kf = 0x1.fb69411e15717p+33 * fexp2(fma(-0x1.18922c0000000p+26, irt, 0x1.e3d70a0000000p+0 * lt));
    const double kb = 0x1.a959ee113f54bp+27 * fexp2(fma(-0x1.30a0b40000000p+24, irt, 0x1.3c48be0000000p+1 * lt));
    const double q = kf * C43 * C1 - kb * C2 * C41;
    cd1 -= q;
    cd2 += q;
    cd41 += q;
    cd43 -= q;
    }
    {  // RP016 (elementary)
    const double kf = 0x1.126108d6b8e49p+89 * fexp2(fma(-0x1.27718b8000000p+29, irt, -0x1.8f5c280000000p+3 * lt));
    const double kb = 0x1.c55129c6bd664p+71 * fexp2(fma(-0x1.fb05740000000p+26, irt, -0x1.87fa440000000p+3 * lt));
    const double q = kf * C43 - kb * C1 * C41;
    cd1 += q;
    cd41 += q;
    cd43 -= q;
    }
    {  // RP018 (elementary)
    const double kf = 0x1.0f3fc749d1dacp+27 * fexp2(fma(-0x1.76c1800000000p+21, irt, 0x1.570a3e0000000p+1 * lt));
    const double kb = 0x1.476320e526456p+23 * fexp2(fma(-0x1.7e57c00000000p+23, irt, 0x1.941fc80000000p+1 * lt));
    const double q = kf * C43 * C4 - kb * C5 * C41;
    cd4 -= q;
    cd5 += q;
    cd41 += q;
    cd43 -= q;
    }
    {  // RK020 (elementary)
    const double kf = 0x1.2f04df965be10p+45 * fexp2(fma(-0x1.34a0ca0000000p+27, irt, 0x1.051eb80000000p+0 * lt));
    const double kb = 0x1.d31cb04023ed2p+33 * fexp2(fma(-0x1.cfa1720000000p+24, irt, 0x1.521ea40000000p+0 * lt));
    const double q = kf * C39 - kb * C1 * C43;
    cd1 += q;
    cd39 -= q;
    cd43 += q;
    }
    {  // RP104 (elementary)
    const double kf = 0x1.bbc88bd8b9e65p+29 * fexp2(fma(-0x1.1b5b100000000p+24, irt, 0x1.9eb8520000000p+0 * lt));
    const double kb = 0x1.20345010bc55dp+50 * fexp2(fma(-0x1.0aeb2a0000000p+28, irt, 0x1.972f760000000p-2 * lt));
    const double q = kf * C39 * C17 - kb * C1 * C37;
    cd1 += q;
    cd17 -= q;
    cd37 += q;
    cd39 -= q;
    }
    {  // RST13 (elementary)
    const double kf = 0x1.b9086c43db9e3p+30 * fexp2(fma(-0x1.86a0000000000p+15, irt, 0x1.28f5c20000000p-2 * lt));
    const double q = kf * C39 * C7;
    cd3 += q;
    cd7 -= q;
    cd10 += q;
    cd39 -= q;
    cd40 += q;
    }
    {  // RI26 (elementary)
    const double kf = 0x1.0e931dd218000p+50 * fexp2(fma(-0x1.67fe340000000p+28, irt, 0.0 * lt));
    const double q = kf * C44;
    cd33 += q;
    cd35 += q;
    cd44 -= q;
    }
    {  // RI07 (elementary)
    const double kf = 0x1.15befe3d95ee1p+32 * fexp2(fma(-0x1.3c39200000000p+24, irt, 0x1.70a3d80000000p-3 * lt));
    const double q = kf * C8 * C44;
    cd7 += q;
    cd8 -= q;
    cd38 += q;
    cd44 -= q;
    }
    {  // RI18 (elementary)
    const double kf = 0x1.42e0878b10e4bp+50 * fexp2(fma(-0x1.8b64b40000000p+26, irt, -0x1.3666660000000p+2 * lt));
    const double q = kf * C44 * C13;
    cd1 = fma(0x1.0000000000000p+1, q, cd1);
    cd13 -= q;
    cd37 += q;
    cd44 -= q;
    }
    {  // RI25 (elementary)
    const double kf = 0x1.0e931dd218000p+51 * fexp2(fma(-0x1.67fe340000000p+28, irt, 0.0 * lt));
    const double q = kf * C44;
    cd17 += q;
    cd26 += q;
    cd35 += q;
    cd44 -= q;
    }
    {  // RI09 (elementary)
    const double kf = 0x1.797cc39ffd60fp+23 * fexp2(fma(0.0, irt, 0x1.0000000000000p+2 * lt));
    const double kb = 0x1.ef8fe54d7e83ap+25 * fexp2(fma(-0x1.8776360000000p+26, irt, 0x1.016bba0000000p+2 * lt));
    const double q = kf * C38 * C13 - kb * C20 * C44;
    cd13 -= q;
    cd20 += q;
    cd38 -= q;
    cd44 += q;
    }
    {  // RI02 (elementary)
    const double kf = 0x1.a13b860000000p+34 * fexp2(fma(-0x1.2064200000000p+23, irt, 0.0 * lt));
    const double kb = 0x1.e400be2b42f88p+30 * fexp2(fma(-0x1.8983b00000000p+26, irt, 0x1.15b5fa0000000p-1 * lt));
    const double q = kf * C38 * C1 - kb * C2 * C44;
    cd1 -= q;
    cd2 += q;
    cd38 -= q;
    cd44 += q;
    }
    {  // RI05 (elementary)
    const double kf = 0x1.f40bd68282e6dp+29 * fexp2(fma(-0x1.1a97c00000000p+22, irt, 0x1.5ae1480000000p+1 * lt));
    const double q = kf * C38 * C3;
    cd3 -= q;
    cd4 += q;
    cd38 -= q;
    cd44 += q;
    }
    {  // RI01 (elementary)
    const double kf = 0x1.2ebaaa96b543dp+90 * fexp2(fma(-0x1.d058120000000p+28, irt, -0x1.e51eb80000000p+3 * lt));
    const double kb = 0x1.5a352271b3f54p+75 * fexp2(fma(-0x1.195d460000000p+27, irt, -0x1.def8380000000p+3 * lt));
    const double q = kf * C38 - kb * C1 * C44;
    cd1 += q;
    cd38 -= q;
    cd44 += q;
    }
    {  // RI06 (elementary)
    const double kf = 0x1.8100000000000p+29 * fexp2(fma(0.0, irt, 0x1.0000000000000p+1 * lt));
    const double kb = 0x1.4187dd99bf1a4p+28 * fexp2(fma(-0x1.2afb0c0000000p+27, irt, 0x1.3826020000000p+1 * lt));
    const double q = kf * C38 * C4 - kb * C5 * C44;
    cd4 -= q;
    cd5 += q;
    cd38 -= q;
    cd44 += q;
    }
    {  // RK110 (elementary)
    const double kf = 0x1.17499de030f63p+27 * fexp2(fma(-0x1.173c600000000p+24, irt, 0x1.828f5c0000000p+1 * lt));
    const double kb = 0x1.5d6fa03001666p+22 * fexp2(fma(-0x1.ef55a00000000p+23, irt, 0x1.bff7280000000p+1 * lt));
    const double q = kf * C37 * C4 - kb * C5 * C42;
    cd4 -= q;
    cd5 += q;
    cd37 -= q;
    cd42 += q;
    }
    {  // RP108 (elementary)
    const double kf = 0x1.126108d6b8e49p+90 * fexp2(fma(-0x1.276ca98000000p+29, irt, -0x1.8f5c280000000p+3 * lt));
    const double kb = 0x1.d5e3b43600da8p+71 * fexp2(fma(-0x1.cee5140000000p+26, irt, -0x1.87e5ca0000000p+3 * lt));
    const double q = kf * C37 - kb * C1 * C42;
    cd1 += q;
    cd37 -= q;
    cd42 += q;
    }
    {  // RK109 (elementary)
    const double kf = 0x1.cc0ba8a45b4a9p+34 * fexp2(fma(-0x1.10dd840000000p+26, irt, 0x1.deb8520000000p+0 * lt));
    const double kb = 0x1.8fc53a5e8ee25p+27 * fexp2(fma(-0x1.87a34c0000000p+22, irt, 0x1.3a0ba20000000p+1 * lt));
    const double q = kf * C37 * C1 - kb * C2 * C42;
    cd1 -= q;
    cd2 += q;
    cd37 -= q;
    cd42 += q;
    }
    {  // RG28 (elementary)
    const double kf = 0x1.bf08eb0000000p+33 * fexp2(fma(-0x1.3265800000000p+21, irt, 0.0 * lt));
    const double kb = 0x1.b9fb5ac9f9a01p+32 * fexp2(fma(-0x1.2fbfbe0000000p+25, irt, -0x1.fe3fd60000000p-5 * lt));
    const double q = kf * C15 * C0 - kb * C0 * C12;
    cd12 += q;
    cd15 -= q;
    }
    {  // R5 (third_body)
    const double kf = 0x1.9e70448800000p+31 * fexp2(fma(0.0, irt, -0x1.0000000000000p+0 * lt));
    const double q = (kf * C1 * C1) * M0();
    cd1 = fma(-0x1.0000000000000p+1, q, cd1);
    cd2 += q;
    }
    {  // R10 (third_body)
    const double kf = 0x1.1272f99b80000p+34 * fexp2(fma(0.0, irt, -0x1.0000000000000p+0 * lt));
    const double q = (kf * C1 * C3) * M1();
    cd1 -= q;
    cd3 -= q;
    cd4 += q;
    }
    {  // R14 (falloff)
    const double kinf_f = 0x1.48f5c74fe0810p+33 * fexp2(fma(0.0, irt, -0x1.7ae1480000000p-2 * lt));
    const double k0_f = 0x1.417095c517ea1p+32 * fexp2(fma(0x1.24a9e00000000p+23, irt, -0x1.28f5c20000000p-1 * lt));
    const double kinf_b = 0x1.836985586c056p+52 * fexp2(fma(-0x1.9994c60000000p+27, irt, -0x1.636b900000000p+0 * lt));
    const double k0_b = 0x1.7a8e47c96d4d4p+51 * fexp2(fma(-0x1.874a280000000p+27, irt, -0x1.992e1e0000000p+0 * lt));
    const double m_ = M1();
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
    const double q = kf * C4 * C4 - kb * C6;
    cd4 = fma(-0x1.0000000000000p+1, q, cd4);
    cd6 += q;
    }
    {  // RG07 (falloff)
    const double kinf_f = 0x1.ad366b951da24p+34 * fexp2(fma(0x1.7a6b000000000p+20, irt, 0x1.b851ec0000000p-2 * lt));
    const double k0_f = 0x1.2328e8c9877bap+40 * fexp2(fma(-0x1.2d83800000000p+21, irt, -0x1.6666660000000p+1 * lt));
    const double m_ = M1();
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
    const double q = kf * C9 * C2;
    cd2 -= q;
    cd9 -= q;
    cd13 += q;
    }
    {  // RG14 (falloff)
    const double kinf_f = 0x1.176592e000000p+39 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double k0_f = 0x1.9324709d7b3d5p+41 * fexp2(fma(-0x1.9853400000000p+22, irt, -0x1.6147ae0000000p+1 * lt));
    const double m_ = M1();
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
    const double q = kf * C12 * C1;
    cd1 -= q;
    cd12 -= q;
    cd13 += q;
    }
    {  // RG24 (falloff)
    const double kinf_f = 0x1.111c906616bd7p+34 * fexp2(fma(-0x1.1feef00000000p+24, irt, 0x1.0000000000000p-1 * lt));
    const double k0_f = 0x1.1812e88a3b07ep+45 * fexp2(fma(-0x1.c508900000000p+24, irt, -0x1.470a3e0000000p+2 * lt));
    const double kinf_b = 0x1.b6aea43f0f007p+56 * fexp2(fma(-0x1.5171860000000p+28, irt, -0x1.3ee43a0000000p+0 * lt));
    const double k0_b = 0x1.c1dd98ab88dd9p+67 * fexp2(fma(-0x1.5bc3200000000p+28, irt, -0x1.b6c34c0000000p+2 * lt));
    const double m_ = M1();
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
    const double q = kf * C12 * C10 - kb * C22;
    cd10 -= q;
    cd12 -= q;
    cd22 += q;
    }
    {  // RG10 (falloff)
    const double kinf_f = 0x1.74876e8000000p+35 * fexp2(fma(0.0, irt, 0.0 * lt));
    const double k0_f = 0x1.cd72ae192db6ap+40 * fexp2(fma(-0x1.ee62800000000p+22, irt, -0x1.deb8520000000p+1 * lt));
    const double kinf_b = 0x1.8fb4cbb0d0cd3p+54 * fexp2(fma(-0x1.2a30e00000000p+28, irt, -0x1.70e3680000000p+0 * lt));
    const double k0_b = 0x1.ef1c822e7b8bap+59 * fexp2(fma(-0x1.31ea6a0000000p+28, irt, -0x1.4b95040000000p+2 * lt));
    const double m_ = M1();
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
    const double q = kf * C9 * C10 - kb * C23;
    cd9 -= q;
    cd10 -= q;
    cd23 += q;
    }
    {  // RG13 (falloff)
    const double kinf_f = 0x1.76aebd8109560p+50 * fexp2(fma(-0x1.5f717b8000000p+28, irt, 0x1.8624de0000000p-2 * lt));
    const double k0_f = 0x1.216c3d614d250p+54 * fexp2(fma(-0x1.622e2a8000000p+28, irt, -0x1.55a1ca0000000p+1 * lt));
    const double m_ = M1();
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
    const double q = kf * C14;
    cd1 += q;
    cd11 += q;
    cd14 -= q;
    }
    {  // RG12 (falloff)
    const double kinf_f = 0x1.477bb84214bc7p+44 * fexp2(fma(-0x1.3fcd628000000p+28, irt, 0x1.a2d0e60000000p-1 * lt));
    const double k0_f = 0x1.b90fc370f0cebp+56 * fexp2(fma(-0x1.52c0758000000p+28, irt, -0x1.06872c0000000p+2 * lt));
    const double m_ = M1();
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
    const double q = kf * C14;
    cd2 += q;
    cd10 += q;
    cd14 -= q;
    }
    {  // RG43 (falloff)
    const double kinf_f = 0x1.e2c7f119a8f26p+42 * fexp2(fma(-0x1.06e0e00000000p+27, irt, 0x1.1a9fbe0000000p-4 * lt));
    const double k0_f = 0x1.24517338b4f55p+53 * fexp2(fma(-0x1.1e43340000000p+27, irt, -0x1.4cdd300000000p+2 * lt));
    const double m_ = M1();
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
    const double q = kf * C24;
    cd1 += q;
    cd14 += q;
    cd24 -= q;
    }
    {  // RG104 (falloff)
    const double kinf_f = 0x1.6bcc41e900000p+37 * fexp2(fma(0.0, irt, -0x1.0000000000000p+0 * lt));
    const double k0_f = 0x1.d410ebe3de347p+47 * fexp2(fma(-0x1.e53ac00000000p+22, irt, -0x1.3333340000000p+2 * lt));
    const double m_ = M1();
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
    const double q = kf * C25 * C1;
    cd1 -= q;
    cd17 += q;
    cd25 -= q;
    }
    {  // RG115 (falloff)
    const double kinf_f = 0x1.5f86fb6c5893cp+35 * fexp2(fma(-0x1.59c3a00000000p+23, irt, 0x1.451eb80000000p+0 * lt));
    const double k0_f = 0x1.b55cde0fc46bap+43 * fexp2(fma(-0x1.e2c9c00000000p+23, irt, -0x1.2a3d700000000p+2 * lt));
    const double kinf_b = 0x1.bc87750d58608p+44 * fexp2(fma(-0x1.2d9c840000000p+27, irt, 0x1.711f0c0000000p+0 * lt));
    const double k0_b = 0x1.148953ea43893p+53 * fexp2(fma(-0x1.362ce60000000p+27, irt, -0x1.1f3d5c0000000p+2 * lt));
    const double m_ = M1();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.b295ea0000000p-3, fexp2(-(-0x1.285504d297b1bp-13 * T)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C17 * C1 - kb * C18;
    cd1 -= q;
    cd17 -= q;
    cd18 += q;
    }
    {  // RG129 (falloff)
    const double kinf_f = 0x1.e83b7f97942bcp+34 * fexp2(fma(-0x1.1da5000000000p+20, irt, 0x1.147ae20000000p-2 * lt));
    const double k0_f = 0x1.6301b0bd56537p+45 * fexp2(fma(-0x1.a7e3a00000000p+23, irt, -0x1.ee147a0000000p+1 * lt));
    const double kinf_b = 0x1.bc2c767d8a9acp+52 * fexp2(fma(-0x1.be05f20000000p+28, irt, 0x1.132f020000000p-3 * lt));
    const double k0_b = 0x1.42f9e418789c5p+63 * fexp2(fma(-0x1.ca276a0000000p+28, irt, -0x1.ff70ce0000000p+1 * lt));
    const double m_ = M1();
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
    const double q = kf * C18 * C1 - kb * C19;
    cd1 -= q;
    cd18 -= q;
    cd19 += q;
    }
    {  // RG155 (falloff)
    const double kinf_f = 0x1.708ea5e351946p+33 * fexp2(fma(-0x1.5a11c00000000p+22, irt, 0x1.75c2900000000p+0 * lt));
    const double k0_f = 0x1.d8cea1c3b83d4p+50 * fexp2(fma(-0x1.7058e00000000p+24, irt, -0x1.a8f5c20000000p+2 * lt));
    const double kinf_b = 0x1.3b83526993a68p+43 * fexp2(fma(-0x1.2b77e20000000p+27, irt, 0x1.56b4640000000p+0 * lt));
    const double k0_b = 0x1.94c21bfdaa83bp+60 * fexp2(fma(-0x1.4eb2700000000p+27, irt, -0x1.b0b94e0000000p+2 * lt));
    const double m_ = M1();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.91a9fc0000000p+0, fexp2(-(0x1.3c3731144eedfp-8 * T)), fc);
    fc = fma(-0x1.2353f80000000p-1, fexp2(-(-0x1.4ac50d8702f03p-13 * T)), fc);
    fc = fma(0x1.0000000000000p+0, fexp2(-(0x1.b7bbc21fd2ed9p+7 * invT)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C19 * C1 - kb * C21;
    cd1 -= q;
    cd19 -= q;
    cd21 += q;
    }
    {  // RG164 (falloff)
    const double kinf_f = 0x1.f8592ae3e59d9p+39 * fexp2(fma(-0x1.9371400000000p+22, irt, -0x1.fae1480000000p-1 * lt));
    const double k0_f = 0x1.744837ad03a96p+53 * fexp2(fma(-0x1.aac9d00000000p+24, irt, -0x1.c51eb80000000p+2 * lt));
    const double m_ = M1();
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
    const double q = kf * C21 * C1;
    cd1 -= q;
    cd21 -= q;
    cd29 += q;
    }
    {  // RG173 (falloff)
    const double kinf_f = 0x1.70e99bf238ae2p+79 * fexp2(fma(-0x1.ac50700000000p+28, irt, -0x1.370a3e0000000p+3 * lt));
    const double k0_f = 0x1.82a3735d09767p+89 * fexp2(fma(-0x1.9552350000000p+28, irt, -0x1.a47ae20000000p+3 * lt));
    const double kinf_b = 0x1.6a536d3035d39p+54 * fexp2(fma(-0x1.ecd6360000000p+25, irt, -0x1.0a447c0000000p+3 * lt));
    const double k0_b = 0x1.7ba3f5f2b0cf4p+64 * fexp2(fma(-0x1.34e45e0000000p+25, irt, -0x1.77b5740000000p+3 * lt));
    const double m_ = M1();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.3851ec0000000p-1, fexp2(-(0x1.d8be0817f5ffep-7 * T)), fc);
    fc = fma(0x1.8f5c280000000p-2, fexp2(-(0x1.8e194a2f1fffep-11 * T)), fc);
    fc = fma(0x1.0000000000000p+0, fexp2(-(0x1.0e815ca995e71p+13 * invT)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C29 - kb * C13 * C13;
    cd13 = fma(0x1.0000000000000p+1, q, cd13);
    cd29 -= q;
    }
    {  // ROX01 (falloff)
    const double kinf_f = 0x1.7626754c0452dp+47 * fexp2(fma(-0x1.3472670000000p+28, irt, 0x1.3d70a40000000p-1 * lt));
    const double k0_f = 0x1.2fa1269593144p+99 * fexp2(fma(-0x1.6784220000000p+28, irt, -0x1.2deb860000000p+4 * lt));
    const double kinf_b = 0x1.033fa9e37a68fp+33 * fexp2(fma(0x1.4260880000000p+21, irt, 0x1.fc0a060000000p-1 * lt));
    const double k0_b = 0x1.a4de029938fd0p+84 * fexp2(fma(-0x1.8467d00000000p+25, irt, -0x1.27f6940000000p+4 * lt));
    const double m_ = M1();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.9168720000000p-4, fexp2(-(0x1.0fb0e4489f08cp-9 * T)), fc);
    fc = fma(0x1.cdd2f20000000p-1, fexp2(-(0x1.081a12d2bfc6bp-8 * T)), fc);
    fc = fma(0x1.0000000000000p+0, fexp2(-(0x1.5bb08363df651p+12 * invT)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);
    const double q = kf * C32 - kb * C1 * C36;
    cd1 += q;
    cd32 -= q;
    cd36 += q;
    }
    {  // R9 (third_body)
    const double kf = 0x1.38a388a43c000p+37 * fexp2(fma(0.0, irt, -0x1.0000000000000p+1 * lt));
    const double kb = 0x1.c8b3c265a295cp+50 * fexp2(fma(-0x1.d926f40000000p+28, irt, -0x1.c0e6080000000p+0 * lt));
    const double q = (kf * C1 * C4 - kb * C5) * M2();
    cd1 -= q;
    cd4 -= q;
    cd5 += q;
    }
    {  // R12 (falloff)
    const double kinf_f = 0x1.28d4aaa8ae8d5p+36 * fexp2(fma(0.0, irt, 0x1.c28f5c0000000p-2 * lt));
    const double k0_f = 0x1.2fdc9732a2fe5p+33 * fexp2(fma(0.0, irt, -0x1.6666660000000p+0 * lt));
    const double m_ = M3();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    double fc = 0.0;
    fc = fma(0x1.0000000000000p-1, fexp2(-(0x1.adf4e5242274dp+33 * T)), fc);
    fc = fma(0x1.0000000000000p-1, fexp2(-(0x1.3d4082b723423p-33 * T)), fc);
    const double l2fc = flog2(fc);
    const double lfc = l2fc * kLog10Of2;
    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);
    const double cco = fma(-kTroeC1, lfc, -kTroeC0);
    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);
    const double q = kf * C1 * C7;
    cd1 -= q;
    cd7 -= q;
    cd8 += q;
    }
    {  // RG51 (falloff)
    const double kinf_f = 0x1.8c30f2efa8b24p+37 * fexp2(fma(0.0, irt, 0x1.70a3d80000000p-3 * lt));
    const double k0_f = 0x1.5101afba610e5p+51 * fexp2(fma(-0x1.43f1b00000000p+24, irt, -0x1.9333340000000p+2 * lt));
    const double kinf_b = 0x1.c6df01f109f46p+54 * fexp2(fma(-0x1.a586fc0000000p+28, irt, 0x1.488ab40000000p-7 * lt));
    const double k0_b = 0x1.82edf56ea9ec6p+68 * fexp2(fma(-0x1.b9c6180000000p+28, irt, -0x1.9e13fe0000000p+2 * lt));
    const double m_ = M4();
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
    const double q = kf * C13 * C1 - kb * C20;
    cd1 -= q;
    cd13 -= q;
    cd20 += q;
    }
    {  // R27 (falloff)
    const double kinf_f = 0x1.9f0a000000000p+23 * fexp2(fma(-0x1.3090c00000000p+23, irt, 0.0 * lt));
    const double k0_f = 0x1.e170d7e16bf09p+34 * fexp2(fma(-0x1.0ba3a00000000p+24, irt, -0x1.651eb80000000p+1 * lt));
    const double m_ = M5();
    const double conc = m_ > 0.0 ? m_ : p_rt;
    const double pr_f = k0_f * conc / fmax(kinf_f, 1.0e-60);
    const double kf = kinf_f * pr_f / (1.0 + pr_f);
    const double q = kf * C10 * C3;
    cd3 -= q;
    cd10 -= q;
    cd16 += q;
    }
    {  // R36 (third_body)
    const double kf = 0x1.5426a92560000p+38 * fexp2(fma(-0x1.0f56e40000000p+26, irt, -0x1.0000000000000p+0 * lt));
    const double kb = 0x1.18d7f8975dd24p+28 * fexp2(fma(-0x1.46ee300000000p+22, irt, -0x1.88d9fa0000000p-1 * lt));
    const double q = (kf * C11 - kb * C1 * C10) * M6();
    cd1 += q;
    cd10 += q;
    cd11 -= q;
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
    cd[36] = cd36;
    cd[37] = cd37;
    cd[38] = cd38;
    cd[39] = cd39;
    cd[40] = cd40;
    cd[41] = cd41;
    cd[42] = cd42;
    cd[43] = cd43;
    cd[44] = cd44;
  }

  // s: [rho*Y (45), rho*T] of this lane's state; f: the right-hand side
  static __device__ __forceinline__ void eval(const double (&s)[46], double P, double (&f)[46]) {
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
    rho += s[36];
    rho += s[37];
    rho += s[38];
    rho += s[39];
    rho += s[40];
    rho += s[41];
    rho += s[42];
    rho += s[43];
    rho += s[44];
    const double T = s[45] / rho;
    const double irho = 1.0 / rho;
    double C[45], cd[45];
    C[0] = s[0] * 0x1.245cd2eb40a46p-5;
    C[1] = s[1] * 0x1.fbefbe72dfd0bp-1;
    C[2] = s[2] * 0x1.fbefbe72dfd0bp-2;
    C[3] = s[3] * 0x1.0000000000000p-4;
    C[4] = s[4] * 0x1.e1a7dc7865ca7p-5;
    C[5] = s[5] * 0x1.c6b4f7f1539dfp-5;
    C[6] = s[6] * 0x1.e1a7dc7865ca7p-6;
    C[7] = s[7] * 0x1.0000000000000p-5;
    C[8] = s[8] * 0x1.f05d519a5a4afp-6;
    C[9] = s[9] * 0x1.3aa42a8f7dbc3p-4;
    C[10] = s[10] * 0x1.24778b96770f5p-5;
    C[11] = s[11] * 0x1.1a4ebab921f45p-5;
    C[12] = s[12] * 0x1.24077255ac595p-4;
    C[13] = s[13] * 0x1.1072f8c06c358p-4;
    C[14] = s[14] * 0x1.10d4897263b9dp-5;
    C[15] = s[15] * 0x1.24077255ac595p-4;
    C[16] = s[16] * 0x1.74476f46bcafbp-6;
    C[17] = s[17] * 0x1.3aa42a8f7dbc3p-5;
    C[18] = s[18] * 0x1.2ee9ec61a82a7p-5;
    C[19] = s[19] * 0x1.24077255ac595p-5;
    C[20] = s[20] * 0x1.fea8d69a8976dp-5;
    C[21] = s[21] * 0x1.19e6472ab1c54p-5;
    C[22] = s[22] * 0x1.85c2db9e52812p-6;
    C[23] = s[23] * 0x1.8f56483547455p-6;
    C[24] = s[24] * 0x1.07f7f2b66042cp-5;
    C[25] = s[25] * 0x1.47503bacf8495p-5;
    C[26] = s[26] * 0x1.a3858cbce86c4p-6;
    C[27] = s[27] * 0x1.40da2e4d27b1cp-6;
    C[28] = s[28] * 0x1.7c434324c92a8p-6;
    C[29] = s[29] * 0x1.1072f8c06c358p-5;
    C[30] = s[30] * 0x1.98f7524ff8349p-6;
    C[31] = s[31] * 0x1.a3858cbce86c4p-7;
    C[32] = s[32] * 0x1.a901a98ec71c1p-7;
    C[33] = s[33] * 0x1.f76d11dd156c1p-7;
    C[34] = s[34] * 0x1.855f43b0f475fp-6;
    C[35] = s[35] * 0x1.47503bacf8495p-6;
    C[36] = s[36] * 0x1.aea2f70276baep-7;
    C[37] = s[37] * 0x1.ff5847037515bp-8;
    C[38] = s[38] * 0x1.1a1bb56fb40cap-7;
    C[39] = s[39] * 0x1.3db7668a51cedp-7;
    C[40] = s[40] * 0x1.67970b936e05bp-7;
    C[41] = s[41] * 0x1.440cf5b39f5c3p-7;
    C[42] = s[42] * 0x1.01b2ff46da78dp-7;
    C[43] = s[43] * 0x1.40da2e4d27b1cp-7;
    C[44] = s[44] * 0x1.1c93ecbd44cc3p-7;
    const bool hi = T > 0x1.f400000000000p+9;
    double cpm = 0.0;
    if (hi) {
      cpm = fma(s[0] * irho, 0x1.28ba9057d1783p+8 * (0x1.769c23b7952d2p+1 + T * (0x1.86106ec5d7fc6p-10 + T * (-0x1.3132bf1b89c39p-21 + T * (0x1.bc128a9b8a724p-34 + T * -0x1.e6a15668d1fd9p-48)))), cpm);
      cpm = fma(s[1] * irho, 0x1.01c2d34acaff7p+13 * (0x1.40000015798eep+1 + T * (-0x1.961a6ec6a1e45p-36 + T * (0x1.230b4c341c642p-46 + T * (-0x1.5d647fbe2e672p-58 + T * 0x1.2d244e9510ba2p-71)))), cpm);
      cpm = fma(s[2] * irho, 0x1.01c2d350092cdp+12 * (0x1.ab2bf6fecf7e5p+1 + T * (-0x1.9e6b00cea2ba4p-15 + T * (0x1.0c24d11e93b22p-21 + T * (-0x1.8adee4a4b6baep-33 + T * 0x1.68bf7de4136dcp-46)))), cpm);
      cpm = fma(s[3] * irho, 0x1.03d2b851eb852p+9 * (0x1.48e2c7b5e1a3dp+1 + T * (-0x1.689a006cdb509p-14 + T * (0x1.6855a2fbdda5cp-25 + T * (-0x1.607823c010ceap-37 + T * 0x1.620b4436bd152p-50)))), cpm);
      cpm = fma(s[4] * irho, 0x1.e8d949731098dp+8 * (0x1.6eaf6f6ecdbe1p+1 + T * (0x1.14f4d0c23ad0ap-10 + T * (-0x1.163020518c34ep-22 + T * (0x1.0c7922a4a2d04p-35 + T * -0x1.7fe9359e80e81p-50)))), cpm);
      cpm = fma(s[5] * irho, 0x1.cd7f5ff609dd0p+8 * (0x1.8459ddac6e07ap+1 + T * (0x1.1d553f9364039p-9 + T * (-0x1.6057d217698d4p-23 + T * (-0x1.aacb906a5f7ccp-34 + T * 0x1.2f01042cd6ffep-46)))), cpm);
      cpm = fma(s[6] * irho, 0x1.e8d94983d7907p+7 * (0x1.0a8f681d1fcb7p+2 + T * (0x1.41abe4bc5704bp-8 + T * (-0x1.fe66ae3495cc5p-20 + T * (0x1.981f91177d524p-32 + T * -0x1.0353229ef325dp-45)))), cpm);
      cpm = fma(s[7] * irho, 0x1.03d2b851eb852p+8 * (0x1.a42a332f575b8p+1 + T * (0x1.84c851ecf574dp-10 + T * (-0x1.96ee255022a3dp-21 + T * (0x1.cca1706e20348p-33 + T * -0x1.8667712a69c18p-46)))), cpm);
      cpm = fma(s[8] * irho, 0x1.f7c6fae7924afp+7 * (0x1.0119fbbf289f6p+2 + T * (0x1.2593e46a1f9dfp-9 + T * (-0x1.5431502070c84p-21 + T * (0x1.f675fa32f618cp-34 + T * -0x1.84c80e71ea191p-47)))), cpm);
      cpm = fma(s[9] * irho, 0x1.3f5713b5bf6a1p+9 * (0x1.70718843050d6p+1 + T * (0x1.fd09d40e9c422p-11 + T * (0x1.3631d6b0442c1p-23 + T * (-0x1.1f62b7f017dbdp-33 + T * 0x1.3d32486a4348dp-46)))), cpm);
      cpm = fma(s[10] * irho, 0x1.28d5af07bfe7ep+8 * (0x1.5b8b33bac2892p+1 + T * (0x1.0e56efb7c8adbp-9 + T * (-0x1.0c1ec8ca156a0p-20 + T * (0x1.f9e45483ed15bp-33 + T * -0x1.6edbeeb572dccp-46)))), cpm);
      cpm = fma(s[11] * irho, 0x1.1e860685553efp+8 * (0x1.62d69c2e745cap+1 + T * (0x1.44dbe8babc438p-8 + T * (-0x1.4d75433aa4a6fp-19 + T * (0x1.43e5261c638b2p-31 + T * -0x1.e08abbb0771a1p-45)))), cpm);
      cpm = fma(s[12] * irho, 0x1.2863e90ff9724p+9 * (0x1.6fe28bbb5f921p+1 + T * (0x1.df4030068403dp-9 + T * (-0x1.7a3607a17a275p-20 + T * (0x1.1e1208519dbd9p-32 + T * -0x1.522e0f41fe4e3p-46)))), cpm);
      cpm = fma(s[13] * irho, 0x1.148494a2b9d3dp+9 * (0x1.7d330e4a459e7p+1 + T * (0x1.7bf7d0ba1fd49p-8 + T * (-0x1.09286973eb98fp-19 + T * (0x1.51e0ab53b03a6p-32 + T * -0x1.42c57f31cb480p-46)))), cpm);
      cpm = fma(s[14] * irho, 0x1.14e7994e1a3f4p+8 * (0x1.c2bc95c7fddb1p+0 + T * (0x1.2d77335291c21p-7 + T * (-0x1.28cb7c4b91fedp-18 + T * (0x1.14a3f4fe94722p-30 + T * -0x1.8e0d9e100cd20p-44)))), cpm);
      cpm = fma(s[15] * irho, 0x1.2863e90ff9724p+9 * (0x1.256183d389aa6p+1 + T * (0x1.3120cfb16b35fp-8 + T * (-0x1.0e0906cfb21aep-19 + T * (0x1.cb7e14e4de1f4p-32 + T * -0x1.31fd42b26d354p-45)))), cpm);
      cpm = fma(s[16] * irho, 0x1.79d6b356da017p+7 * (0x1.edc1423f95973p+1 + T * (0x1.214cd7e62db66p-8 + T * (-0x1.29446e529e95bp-19 + T * (0x1.1fcab1b9912a3p-31 + T * -0x1.a937326a2284cp-45)))), cpm);
      cpm = fma(s[17] * irho, 0x1.3f5713ad5bee4p+8 * (0x1.0971c7ee6bae0p+2 + T * (0x1.86b42b3f9ab1ep-8 + T * (-0x1.3e7de3eb387edp-19 + T * (0x1.00f66a3bafde2p-31 + T * -0x1.455f2b475f023p-45)))), cpm);
      cpm = fma(s[18] * irho, 0x1.33700096feb4ap+8 * (0x1.8224031487768p+1 + T * (0x1.52803e497ede9p-7 + T * (-0x1.3a1fef6b5677dp-18 + T * (0x1.17b98c3c9686ep-30 + T * -0x1.847bd21d4a0a4p-44)))), cpm);
      cpm = fma(s[19] * irho, 0x1.2863e90ff9724p+8 * (0x1.049f4a5d9c3d6p+1 + T * (0x1.dfe6a5720731ep-7 + T * (-0x1.c25a4ed3d3908p-18 + T * (0x1.94aeec0be93f2p-30 + T * -0x1.1b109c49479cdp-43)))), cpm);
      cpm = fma(s[20] * irho, 0x1.03249374bc6a8p+9 * (0x1.a73c320a693a8p+0 + T * (0x1.488ac88f5e28fp-7 + T * (-0x1.bd25ef0359a5ep-19 + T * (0x1.26ef4a1545f72p-31 + T * -0x1.1b7421c730b17p-45)))), cpm);
      cpm = fma(s[21] * irho, 0x1.1e1c0389f83bep+8 * (0x1.f4645cf6d1024p+0 + T * (0x1.1d0972c8defc6p-6 + T * (-0x1.0bd56e41b638fp-17 + T * (0x1.e1a27cc16cb18p-30 + T * -0x1.50f67ed791cc7p-43)))), cpm);
      cpm = fma(s[22] * irho, 0x1.8b94f63800219p+7 * (0x1.20b91864fbad3p+2 + T * (0x1.2707a64c0b6f9p-7 + T * (-0x1.17cdaf120e12fp-18 + T * (0x1.fb9d615c62415p-31 + T * -0x1.65f69aff87e86p-44)))), cpm);
      cpm = fma(s[23] * irho, 0x1.954cff43419e3p+7 * (0x1.683486198a14cp+2 + T * (0x1.0bbca21f5e9bfp-8 + T * (-0x1.abbd5f8926da2p-20 + T * (0x1.3abf2c56d8d5fp-32 + T * -0x1.5d9ed3d5e2c0fp-46)))), cpm);
      cpm = fma(s[24] * irho, 0x1.0be922424a277p+8 * (0x1.d8a944f2ce3e4p+1 + T * (0x1.1b4df55708be3p-7 + T * (-0x1.f773c3714a914p-19 + T * (0x1.b0c96ce8203e2p-31 + T * -0x1.24153561cd7f6p-44)))), cpm);
      cpm = fma(s[25] * irho, 0x1.4c3397bb73083p+8 * (0x1.957aaf1dba502p+1 + T * (0x1.377101463a6fcp-8 + T * (-0x1.ed598482ed583p-20 + T * (0x1.4e75f1b05c789p-32 + T * -0x1.3f4630515edadp-46)))), cpm);
      cpm = fma(s[26] * irho, 0x1.a9c96fa82e87dp+7 * (0x1.898bb8a5a3682p+2 + T * (0x1.3212e5c078a87p-7 + T * (-0x1.f76409d296ab1p-19 + T * (0x1.7b6addd20d988p-31 + T * -0x1.9f130253a1242p-45)))), cpm);
      cpm = fma(s[27] * irho, 0x1.45a4d67fd3f5bp+7 * (0x1.d0361814f4aecp+2 + T * (0x1.87d7af23d086fp-7 + T * (-0x1.6179105e26871p-18 + T * (0x1.2e50dd402de5cp-30 + T * -0x1.8e203138592dbp-44)))), cpm);
      cpm = fma(s[28] * irho, 0x1.81f10d173fb7ap+7 * (0x1.02071e6cd2913p+3 + T * (0x1.01f6d02b7c04bp-6 + T * (-0x1.5bc8d10e059f3p-18 + T * (0x1.9b10de3c923b6p-31 + T * -0x1.5b2ceb945d02cp-45)))), cpm);
      cpm = fma(s[29] * irho, 0x1.148494a2b9d3dp+8 * (0x1.1266d373affb0p+0 + T * (0x1.634a9ae4e575dp-6 + T * (-0x1.50674e48c90f9p-17 + T * (0x1.304e6c1a9e602p-29 + T * -0x1.abd9357b132f9p-43)))), cpm);
      cpm = fma(s[30] * irho, 0x1.9f12d9cf13cefp+7 * (0x1.6844fda07f3bfp+1 + T * (0x1.2ff69d12bb67ap-6 + T * (-0x1.40742cb99df7cp-17 + T * (0x1.49c96202a850fp-29 + T * -0x1.0b6277075476ap-42)))), cpm);
      cpm = fma(s[31] * irho, 0x1.a9c96fa82e87dp+6 * (-0x1.a6617a5d2d1b8p-3 + T * (0x1.7c3587c3a5a91p-5 + T * (-0x1.d1d34921ec523p-16 + T * (0x1.0f114e0097577p-27 + T * -0x1.e457b37c410e3p-41)))), cpm);
      cpm = fma(s[32] * irho, 0x1.af5a836eb4e98p+6 * (0x1.615262ce5664cp+0 + T * (0x1.4afba7509d6e9p-5 + T * (-0x1.966df67d59e07p-16 + T * (0x1.d9497ceb0d2b7p-28 + T * -0x1.a6c0db72a09e5p-41)))), cpm);
      cpm = fma(s[33] * irho, 0x1.fef1b93037d63p+6 * (0x1.0dbccff4ca6cdp+2 + T * (0x1.bd5fbfaabbb01p-6 + T * (-0x1.bedaea5c5a06bp-17 + T * (0x1.a8a8b6f9d257dp-29 + T * -0x1.38dd6b9a13bc8p-42)))), cpm);
      cpm = fma(s[34] * irho, 0x1.8b2fe175d13d7p+7 * (0x1.e304cbb91de5cp-2 + T * (0x1.da56952f74035p-6 + T * (-0x1.06bbf817964e9p-16 + T * (0x1.1abdda60836a8p-28 + T * -0x1.dc571b665fffdp-42)))), cpm);
      cpm = fma(s[35] * irho, 0x1.4c3397bb73083p+7 * (0x1.3844cbbc5687fp+3 + T * (0x1.f098c20ad452dp-9 + T * (0x1.48b7ad22b4b01p-22 + T * (-0x1.5c5b043d5fc7cp-31 + T * 0x1.fc9776606b4d0p-44)))), cpm);
      cpm = fma(s[36] * irho, 0x1.b51158b827fa2p+6 * (0x1.7e3b62413db7fp+1 + T * (0x1.1497c9ab7243ap-5 + T * (-0x1.4ff1bbec5496ap-16 + T * (0x1.837a30524ba65p-28 + T * -0x1.5766dcb184e46p-41)))), cpm);
      cpm = fma(s[37] * irho, 0x1.037d9b6c01b0ep+6 * (0x1.c4acde19fc2a9p+0 + T * (0x1.1a45ef20d54fbp-4 + T * (-0x1.5b8f028203f25p-15 + T * (0x1.952685e7590bap-27 + T * -0x1.69f7f2ba9e932p-40)))), cpm);
      cpm = fma(s[38] * irho, 0x1.1e523e4e19688p+6 * (0x1.2793bc5fed258p+0 + T * (0x1.0bf86109b70c4p-4 + T * (-0x1.4941d47494f93p-15 + T * (0x1.7f58fd89a5ea2p-27 + T * -0x1.5640c191d31a3p-40)))), cpm);
      cpm = fma(s[39] * irho, 0x1.427612472a610p+6 * (0x1.7ebfa91811c4ap+2 + T * (0x1.808ef9036bd83p-5 + T * (-0x1.c0962e1e35445p-16 + T * (0x1.f57fe5096dd33p-28 + T * -0x1.b216377d340d7p-41)))), cpm);
      cpm = fma(s[40] * irho, 0x1.6cf5cd62f4c1ep+6 * (0x1.a676af33dfab7p+1 + T * (0x1.8942e6d1d3136p-5 + T * (-0x1.d3265e0944fbdp-16 + T * (0x1.096280c15fae5p-27 + T * -0x1.d1a5795006dc6p-41)))), cpm);
      cpm = fma(s[41] * irho, 0x1.48e3d91c66681p+6 * (0x1.cf3d5e900342dp+2 + T * (0x1.3a6b3bb31588dp-5 + T * (-0x1.6f2bac59222d5p-16 + T * (0x1.9a5db7b1d766ap-28 + T * -0x1.62db386060849p-41)))), cpm);
      cpm = fma(s[42] * irho, 0x1.058c366871d96p+6 * (0x1.9d4d598f935b6p+1 + T * (0x1.0290e103fe76cp-4 + T * (-0x1.3f4171a96c4d1p-15 + T * (0x1.74a5353c9c597p-27 + T * -0x1.4d1ac451ac8a7p-40)))), cpm);
      cpm = fma(s[43] * irho, 0x1.45a4d67fd3f5bp+6 * (0x1.742c5116c8ef4p+2 + T * (0x1.6929c15c90ab8p-5 + T * (-0x1.a6e04ec509c0ep-16 + T * (0x1.da5a809896006p-28 + T * -0x1.9bbacf12d5814p-41)))), cpm);
      cpm = fma(s[44] * irho, 0x1.20d3e75f1f4a5p+6 * (0x1.d3f701135069dp+1 + T * (0x1.d6e2126028298p-5 + T * (-0x1.1f9ee6937d09fp-15 + T * (0x1.4d62a00d91813p-27 + T * -0x1.28a2e9b5c9733p-40)))), cpm);
    } else {
      cpm = fma(s[0] * irho, 0x1.28ba9057d1783p+8 * (0x1.a63b0c4588a05p+1 + T * (0x1.712969da04050p-10 + T * (-0x1.09f7a2b098bd4p-18 + T * (0x1.83ae94da0fe59p-28 + T * -0x1.581526048e0d6p-39)))), cpm);
      cpm = fma(s[1] * irho, 0x1.01c2d34acaff7p+13 * (0x1.4000000000000p+1 + T * (0x1.8d112bff6d580p-41 + T * (-0x1.1fa470055807fp-49 + T * (0x1.538a620b2373fp-59 + T * -0x1.1863cffe0b329p-70)))), cpm);
      cpm = fma(s[2] * irho, 0x1.01c2d350092cdp+12 * (0x1.2c130ac9b2911p+1 + T * (0x1.058175d02a941p-7 + T * (-0x1.46ca05831775cp-16 + T * (0x1.5a4c582f87e3dp-26 + T * -0x1.03862939e564dp-37)))), cpm);
      cpm = fma(s[3] * irho, 0x1.03d2b851eb852p+9 * (0x1.9589c6bdbf12dp+1 + T * (-0x1.add3ae5787a18p-9 + T * (0x1.bdcef845b6ae0p-18 + T * (-0x1.a51e14d5c0503p-28 + T * 0x1.2954967e1b470p-39)))), cpm);
      cpm = fma(s[4] * irho, 0x1.e8d949731098dp+8 * (0x1.080501d23d242p+2 + T * (-0x1.a6c41f4a374cap-9 + T * (0x1.b6101eb7dedbep-18 + T * (-0x1.8e78ee8164a9cp-28 + T * 0x1.2240d8be85bd5p-39)))), cpm);
      cpm = fma(s[5] * irho, 0x1.cd7f5ff609dd0p+8 * (0x1.0cb686e536fbfp+2 + T * (-0x1.0aeb63b84c925p-9 + T * (0x1.b593a7c039b70p-18 + T * (-0x1.7921667072d59p-28 + T * 0x1.f2c47bce627b1p-40)))), cpm);
      cpm = fma(s[6] * irho, 0x1.e8d94983d7907p+7 * (0x1.11abd48f63e0ap+2 + T * (-0x1.1c98643a78c6ap-11 + T * (0x1.18be22e62f026p-16 + T * (-0x1.72b101d35ae59p-26 + T * 0x1.2f72fba30b7c2p-37)))), cpm);
      cpm = fma(s[7] * irho, 0x1.03d2b851eb852p+8 * (0x1.e42787ae5fa45p+1 + T * (-0x1.88c9b66c8c0dfp-9 + T * (0x1.4a6bae1fdae75p-17 + T * (-0x1.4ca5927ada53cp-27 + T * 0x1.c883a18b02bcdp-39)))), cpm);
      cpm = fma(s[8] * irho, 0x1.f7c6fae7924afp+7 * (0x1.1350a899bcaa1p+2 + T * (-0x1.373d054674594p-8 + T * (0x1.62fa28e3a8ea6p-16 + T * (-0x1.a110b0905e0fcp-26 + T * 0x1.46f1288fc5c1cp-37)))), cpm);
      cpm = fma(s[9] * irho, 0x1.3f5713b5bf6a1p+9 * (0x1.beb24fde64a4cp+1 + T * (0x1.5390f0ed10ec5p-12 + T * (-0x1.c5628dbdf8e58p-20 + T * (0x1.b29b14b88d49cp-29 + T * -0x1.8bc782bbe23bbp-40)))), cpm);
      cpm = fma(s[10] * irho, 0x1.28d5af07bfe7ep+8 * (0x1.ca2e271a4b2fdp+1 + T * (-0x1.400048c1ba1b0p-11 + T * (0x1.10f2f2ddb1673p-20 + T * (0x1.f2a1bae3bf93ap-31 + T * -0x1.fd254e88ba403p-41)))), cpm);
      cpm = fma(s[11] * irho, 0x1.1e860685553efp+8 * (0x1.0e27e8a748d9cp+2 + T * (-0x1.a9301251f436fp-9 + T * (0x1.ce60d2a2b7dfep-17 + T * (-0x1.c97ac8618dbf3p-27 + T * 0x1.313cda197894cp-38)))), cpm);
      cpm = fma(s[12] * irho, 0x1.2863e90ff9724p+9 * (0x1.e19f746480de1p+1 + T * (0x1.fbf7d158743a2p-11 + T * (0x1.771ffa66e83e0p-19 + T * (-0x1.08a1f3bb46844p-28 + T * 0x1.daf7390cac908p-40)))), cpm);
      cpm = fma(s[13] * irho, 0x1.148494a2b9d3dp+9 * (0x1.d41e76e38c2bfp+1 + T * (0x1.16bcc8dd4edc2p-9 + T * (0x1.6e4e659e7b1a3p-18 + T * (-0x1.c6cada0b83d8bp-28 + T * 0x1.5b0478af296dap-39)))), cpm);
      cpm = fma(s[14] * irho, 0x1.14e7994e1a3f4p+8 * (0x1.32cc5c2ed4ffap+2 + T * (-0x1.44ad209405144p-7 + T * (0x1.391462ecfccf9p-15 + T * (-0x1.45cdb600576d1p-25 + T * 0x1.cfa240d78baa9p-37)))), cpm);
      cpm = fma(s[15] * irho, 0x1.2863e90ff9724p+9 * (0x1.0cb5ee035346ap+2 + T * (-0x1.36326518bab75p-9 + T * (0x1.14409b5702698p-17 + T * (-0x1.cb9b5a07323d1p-28 + T * 0x1.1179431daea17p-39)))), cpm);
      cpm = fma(s[16] * irho, 0x1.79d6b356da017p+7 * (0x1.2daac1343d496p+1 + T * (0x1.266842a5bf315p-7 + T * (-0x1.de0de0090effep-18 + T * (0x1.51fd10511d1a8p-29 + T * -0x1.43952648a136cp-43)))), cpm);
      cpm = fma(s[17] * irho, 0x1.3f5713ad5bee4p+8 * (0x1.9e0b72c73f3bap-1 + T * (0x1.7ec17f28e481ap-6 + T * (-0x1.29f09105c533cp-15 + T * (0x1.e14c5845a203fp-26 + T * -0x1.2b17c43e837e8p-37)))), cpm);
      cpm = fma(s[18] * irho, 0x1.33700096feb4ap+8 * (0x1.9b3219c31fa4ep+1 + T * (0x1.8d17f1df63fcdp-10 + T * (0x1.b2e198409699cp-16 + T * (-0x1.3339cad4b897fp-25 + T * 0x1.02dedc9720552p-36)))), cpm);
      cpm = fma(s[19] * irho, 0x1.2863e90ff9724p+8 * (0x1.fac71d356ff96p+1 + T * (-0x1.f0244a6c1abf8p-8 + T * (0x1.defb3b4522b25p-15 + T * (-0x1.2908fcd07cb16p-24 + T * 0x1.dac91dbd28c88p-36)))), cpm);
      cpm = fma(s[20] * irho, 0x1.03249374bc6a8p+9 * (0x1.498b184c7d064p+2 + T * (-0x1.bfaed90747e6dp-7 + T * (0x1.9c42ed08644bap-15 + T * (-0x1.9ff6fd7e220d5p-25 + T * 0x1.251784fcaea40p-36)))), cpm);
      cpm = fma(s[21] * irho, 0x1.1e1c0389f83bep+8 * (0x1.139d223a3c91dp+2 + T * (-0x1.125f4e7e42173p-8 + T * (0x1.a1089ad91c191p-15 + T * (-0x1.0152aabf3f38cp-24 + T * 0x1.958406c58ed2fp-36)))), cpm);
      cpm = fma(s[22] * irho, 0x1.8b94f63800219p+7 * (0x1.116315790e08dp+1 + T * (0x1.28dc0ec708b6bp-6 + T * (-0x1.23d5df074d80ap-16 + T * (0x1.410e7ab1ff68dp-27 + T * -0x1.1b86c153f96acp-39)))), cpm);
      cpm = fma(s[23] * irho, 0x1.954cff43419e3p+7 * (0x1.203868265a06ep+1 + T * (0x1.2142867388492p-6 + T * (-0x1.8e1bb67756fd6p-16 + T * (0x1.28cb9772e0568p-26 + T * -0x1.64859c0d2ee1dp-38)))), cpm);
      cpm = fma(s[24] * irho, 0x1.0be922424a277p+8 * (0x1.ee93ebafbbefep+1 + T * (0x1.6ec96e6bebfdfp-8 + T * (0x1.8e23514e314c1p-18 + T * (-0x1.672b5483bb261p-27 + T * 0x1.337d06dd584f1p-38)))), cpm);
      cpm = fma(s[25] * irho, 0x1.4c3397bb73083p+8 * (0x1.71e04a987f933p+1 + T * (0x1.b76ae82ebca6cp-7 + T * (-0x1.ddc391c23021ap-16 + T * (0x1.fa727902a68efp-26 + T * -0x1.80ad12085942bp-37)))), cpm);
      cpm = fma(s[26] * irho, 0x1.a9c96fa82e87dp+7 * (0x1.672a8234a31fdp+0 + T * (0x1.ee6ce841ba8dfp-6 + T * (-0x1.4e3e59ef470bdp-15 + T * (0x1.f849e52505b67p-26 + T * -0x1.324c95e6b90dep-37)))), cpm);
      cpm = fma(s[27] * irho, 0x1.45a4d67fd3f5bp+7 * (-0x1.22f59a4800a4ep-5 + T * (0x1.60ac2d434fce0p-5 + T * (-0x1.e2f4e4942c6d4p-15 + T * (0x1.653dab8ab0d77p-25 + T * -0x1.a8dab3f26eac7p-37)))), cpm);
      cpm = fma(s[28] * irho, 0x1.81f10d173fb7ap+7 * (0x1.b69ad42c3c9efp+0 + T * (0x1.a0950b6a6c5a7p-6 + T * (0x1.a8584c6fbe8a6p-20 + T * (-0x1.38e5016099350p-26 + T * 0x1.3698f1640fc84p-37)))), cpm);
      cpm = fma(s[29] * irho, 0x1.148494a2b9d3dp+8 * (0x1.12a6b4b528ec3p+2 + T * (-0x1.688c91f95b2dfp-8 + T * (0x1.f6d86463b6ba0p-15 + T * (-0x1.3048b11b68ad6p-24 + T * 0x1.d8ad50563705bp-36)))), cpm);
      cpm = fma(s[30] * irho, 0x1.9f12d9cf13cefp+7 * (0x1.763575adac203p+0 + T * (0x1.9317093d07cbcp-6 + T * (-0x1.3f229ba9c106ap-16 + T * (0x1.279e5def01329p-27 + T * -0x1.d54d1432e73e0p-40)))), cpm);
      cpm = fma(s[31] * irho, 0x1.a9c96fa82e87dp+6 * (-0x1.60ff53bd6c5cap+2 + T * (0x1.0860ad13f4d48p-4 + T * (-0x1.72468e97f0d63p-15 + T * (0x1.00e9750c5d629p-27 + T * 0x1.b4aef6a6981f7p-39)))), cpm);
      cpm = fma(s[32] * irho, 0x1.af5a836eb4e98p+6 * (-0x1.38195eab8701ep+2 + T * (0x1.00bd599769f74p-4 + T * (-0x1.98dcd80b074d6p-15 + T * (0x1.e4e479f514788p-27 + T * 0x1.23e65d32af969p-41)))), cpm);
      cpm = fma(s[33] * irho, 0x1.fef1b93037d63p+6 * (-0x1.d8385e2ad89bcp+2 + T * (0x1.8e4aac1b8863fp-4 + T * (-0x1.63a21b41e5384p-13 + T * (0x1.460731e1085dfp-23 + T * -0x1.c26d259607371p-35)))), cpm);
      cpm = fma(s[34] * irho, 0x1.8b2fe175d13d7p+7 * (-0x1.2c7f737f5dec1p-9 + T * (0x1.fc54ec2f57755p-6 + T * (-0x1.186f0b100b85cp-16 + T * (0x1.049384aad25cbp-29 + T * 0x1.5fb9aac7a71a0p-40)))), cpm);
      cpm = fma(s[35] * irho, 0x1.4c3397bb73083p+7 * (0x1.62f85428e5ec2p-3 + T * (0x1.73e002f9486fap-5 + T * (-0x1.323c730520ed8p-14 + T * (0x1.ff513db49caa2p-25 + T * -0x1.49d39c160df99p-36)))), cpm);
      cpm = fma(s[36] * irho, 0x1.b51158b827fa2p+6 * (-0x1.bb2c88b499fb1p+1 + T * (0x1.d63c00365bb1bp-5 + T * (-0x1.9d8b964d264dap-15 + T * (0x1.479629cdfcee1p-26 + T * -0x1.130b555d86772p-39)))), cpm);
      cpm = fma(s[37] * irho, 0x1.037d9b6c01b0ep+6 * (-0x1.172dd75917c95p+3 + T * (0x1.af9ec0c249de6p-4 + T * (-0x1.504307a4e92d6p-14 + T * (0x1.7775892d3f086p-26 + T * 0x1.8fe1c739182fap-40)))), cpm);
      cpm = fma(s[38] * irho, 0x1.1e523e4e19688p+6 * (-0x1.03fbb9a4a6e8ep+3 + T * (0x1.9072c60f26353p-4 + T * (-0x1.325df72b41c32p-14 + T * (0x1.437d056bfaa1ep-26 + T * 0x1.0300f3e807b17p-39)))), cpm);
      cpm = fma(s[39] * irho, 0x1.427612472a610p+6 * (-0x1.93d68de0feb30p+2 + T * (0x1.857de9ab4df8cp-4 + T * (-0x1.90d96f509321dp-14 + T * (0x1.aac13c9bdfc98p-25 + T * -0x1.66263ee528523p-37)))), cpm);
      cpm = fma(s[40] * irho, 0x1.6cf5cd62f4c1ep+6 * (-0x1.848391dade5d7p+2 + T * (0x1.561939bd040fbp-4 + T * (-0x1.371770a3b7c95p-14 + T * (0x1.0cff425bb551dp-25 + T * -0x1.2a21c22f075a8p-38)))), cpm);
      cpm = fma(s[41] * irho, 0x1.48e3d91c66681p+6 * (-0x1.1b5d695ce5df1p+2 + T * (0x1.56b310ec94f1cp-4 + T * (-0x1.6cf2f58f7e5bfp-14 + T * (0x1.93f8e91870774p-25 + T * -0x1.663c964ee2b15p-37)))), cpm);
      cpm = fma(s[42] * irho, 0x1.058c366871d96p+6 * (-0x1.00dea94dec9cfp+3 + T * (0x1.a5942dec43d7fp-4 + T * (-0x1.5deb4664a0a76p-14 + T * (0x1.d386683ca0c59p-26 + T * -0x1.97e409514e1edp-41)))), cpm);
      cpm = fma(s[43] * irho, 0x1.45a4d67fd3f5bp+6 * (-0x1.4d76b09635611p+2 + T * (0x1.6287b313f364dp-4 + T * (-0x1.626bfcd3f1a1ep-14 + T * (0x1.6a6d582dd42b8p-25 + T * -0x1.1f5fc1903a77bp-37)))), cpm);
      cpm = fma(s[44] * irho, 0x1.20d3e75f1f4a5p+6 * (-0x1.17944e81176cbp+3 + T * (0x1.a79d720519df1p-4 + T * (-0x1.834fd4f2f7ffep-14 + T * (0x1.42a85cabc7268p-25 + T * -0x1.360c63a20f300p-38)))), cpm);
    }
    rates(C, T, P, cd);
    f[0] = cd[0] * 0x1.c051ec0000000p+4;
    f[1] = cd[1] * 0x1.020c4a0000000p+0;
    f[2] = cd[2] * 0x1.020c4a0000000p+1;
    f[3] = cd[3] * 0x1.0000000000000p+4;
    f[4] = cd[4] * 0x1.1020c40000000p+4;
    f[5] = cd[5] * 0x1.20418a0000000p+4;
    f[6] = cd[6] * 0x1.1020c40000000p+5;
    f[7] = cd[7] * 0x1.0000000000000p+5;
    f[8] = cd[8] * 0x1.0810620000000p+5;
    f[9] = cd[9] * 0x1.a093740000000p+3;
    f[10] = cd[10] * 0x1.c028f60000000p+4;
    f[11] = cd[11] * 0x1.d049ba0000000p+4;
    f[12] = cd[12] * 0x1.c0d4fe0000000p+3;
    f[13] = cd[13] * 0x1.e116880000000p+3;
    f[14] = cd[14] * 0x1.e06a7e0000000p+4;
    f[15] = cd[15] * 0x1.c0d4fe0000000p+3;
    f[16] = cd[16] * 0x1.60147a0000000p+5;
    f[17] = cd[17] * 0x1.a093740000000p+4;
    f[18] = cd[18] * 0x1.b0b43a0000000p+4;
    f[19] = cd[19] * 0x1.c0d4fe0000000p+4;
    f[20] = cd[20] * 0x1.00ac080000000p+4;
    f[21] = cd[21] * 0x1.d0f5c20000000p+4;
    f[22] = cd[22] * 0x1.5049ba0000000p+5;
    f[23] = cd[23] * 0x1.4839580000000p+5;
    f[24] = cd[24] * 0x1.f08b440000000p+4;
    f[25] = cd[25] * 0x1.9072b00000000p+4;
    f[26] = cd[26] * 0x1.386e980000000p+5;
    f[27] = cd[27] * 0x1.9883120000000p+5;
    f[28] = cd[28] * 0x1.58b0200000000p+5;
    f[29] = cd[29] * 0x1.e116880000000p+4;
    f[30] = cd[30] * 0x1.407efa0000000p+5;
    f[31] = cd[31] * 0x1.386e980000000p+6;
    f[32] = cd[32] * 0x1.3466660000000p+6;
    f[33] = cd[33] * 0x1.045c280000000p+6;
    f[34] = cd[34] * 0x1.509fbe0000000p+5;
    f[35] = cd[35] * 0x1.9072b00000000p+5;
    f[36] = cd[36] * 0x1.305e360000000p+6;
    f[37] = cd[37] * 0x1.0053f80000000p+7;
    f[38] = cd[38] * 0x1.d09db20000000p+6;
    f[39] = cd[39] * 0x1.9c8b440000000p+6;
    f[40] = cd[40] * 0x1.6c81060000000p+6;
    f[41] = cd[41] * 0x1.947ae20000000p+6;
    f[42] = cd[42] * 0x1.fc9fbe0000000p+6;
    f[43] = cd[43] * 0x1.9883120000000p+6;
    f[44] = cd[44] * 0x1.cc95820000000p+6;
    double tmp = 0.0;
    if (hi) {
      tmp = fma(-(0x1.28ba9057d1783p+8 * (T * (0x1.769c23b7952d2p+1 + T * (0x1.86106ec5d7fc6p-11 + T * (-0x1.96ee5424b7af6p-23 + T * (0x1.bc128a9b8a724p-36 + T * -0x1.854ddeba4197bp-50)))) + -0x1.cd661b089a027p+9)), f[0], tmp);
      tmp = fma(-(0x1.01c2d34acaff7p+13 * (T * (0x1.40000015798eep+1 + T * (-0x1.961a6ea91e1b0p-37 + T * (0x1.840f104982ce0p-48 + T * (-0x1.5d647fca8f878p-60 + T * 0x1.e1d3b0ee8129dp-74)))) + 0x1.8e06a3bcd35a8p+14)), f[1], tmp);
      tmp = fma(-(0x1.01c2d350092cdp+12 * (T * (0x1.ab2bf6fecf7e5p+1 + T * (-0x1.9e6b00c08fd91p-16 + T * (0x1.65866c34c762ap-23 + T * (-0x1.8adee4a4b6baep-35 + T * 0x1.2099318342be3p-48)))) + -0x1.db14578e5c4ebp+9)), f[2], tmp);
      tmp = fma(-(0x1.03d2b851eb852p+9 * (T * (0x1.48e2c7b5e1a3dp+1 + T * (-0x1.689a0073e4c12p-15 + T * (0x1.e0722e91f065fp-27 + T * (-0x1.607823b4427e2p-39 + T * 0x1.1b3c369230ddcp-52)))) + 0x1.c88650ff97247p+14)), f[3], tmp);
      tmp = fma(-(0x1.e8d949731098dp+8 * (T * (0x1.6eaf6f6ecdbe1p+1 + T * (0x1.14f4d0c23ad0ap-11 + T * (-0x1.72ead5bfa9624p-24 + T * (0x1.0c7922a4a2d04p-37 + T * -0x1.3320f7b200b9ap-52)))) + 0x1.d0db729b280f1p+11)), f[4], tmp);
      tmp = fma(-(0x1.cd7f5ff609dd0p+8 * (T * (0x1.8459ddac6e07ap+1 + T * (0x1.1d553f9364039p-10 + T * (-0x1.d5ca6d6fbef3fp-25 + T * (-0x1.aacb905b9d982p-36 + T * 0x1.e4ce6d148b330p-49)))) + -0x1.d4d1303afb7e9p+14)), f[5], tmp);
      tmp = fma(-(0x1.e8d94983d7907p+7 * (T * (0x1.0a8f681d1fcb7p+2 + T * (0x1.41abe4bc5704bp-9 + T * (-0x1.544474260f258p-21 + T * (0x1.981f91177d524p-34 + T * -0x1.9eeb6a97eb6fbp-48)))) + -0x1.1717269ad42c4p+14)), f[6], tmp);
      tmp = fma(-(0x1.03d2b851eb852p+8 * (T * (0x1.a42a332f575b8p+1 + T * (0x1.84c851ecf574dp-11 + T * (-0x1.0f496e2f6b32bp-22 + T * (0x1.cca17066bf423p-35 + T * -0x1.3852c0eebb013p-48)))) + -0x1.101d4b48d3ae7p+10)), f[7], tmp);
      tmp = fma(-(0x1.f7c6fae7924afp+7 * (T * (0x1.0119fbbf289f6p+2 + T * (0x1.2593e454221e1p-10 + T * (-0x1.c597157493eb4p-23 + T * (0x1.f675fa32f618cp-36 + T * -0x1.370671f4bb474p-49)))) + 0x1.bf6d462c343b7p+6)), f[8], tmp);
      tmp = fma(-(0x1.3f5713b5bf6a1p+9 * (T * (0x1.70718843050d6p+1 + T * (0x1.fd09d405d0756p-12 + T * (0x1.9d97c8efd3589p-25 + T * (-0x1.1f62b7f778ce2p-35 + T * 0x1.fb83a7106ba7cp-49)))) + 0x1.15646fb7e9100p+16)), f[9], tmp);
      tmp = fma(-(0x1.28d5af07bfe7ep+8 * (T * (0x1.5b8b33bac2892p+1 + T * (0x1.0e56efcdc62d9p-10 + T * (-0x1.657e6113731d3p-22 + T * (0x1.f9e45483ed15bp-35 + T * -0x1.257cbef78f170p-48)))) + -0x1.ba3efaacd9e84p+13)), f[10], tmp);
      tmp = fma(-(0x1.1e860685553efp+8 * (T * (0x1.62d69c2e745cap+1 + T * (0x1.44dbe8babc438p-9 + T * (-0x1.bc9c59a08596ap-21 + T * (0x1.43e5262ed5e8fp-33 + T * -0x1.806efc81153b4p-47)))) + 0x1.f57d617c1bda5p+11)), f[11], tmp);
      tmp = fma(-(0x1.2863e90ff9724p+9 * (T * (0x1.6fe28bbb5f921p+1 + T * (0x1.df4030068403dp-10 + T * (-0x1.f8480a32a419ap-22 + T * (0x1.1e12084ded447p-34 + T * -0x1.0e8b3f67fea4fp-48)))) + 0x1.696f353f7ced9p+15)), f[12], tmp);
      tmp = fma(-(0x1.148494a2b9d3dp+9 * (T * (0x1.7d330e4a459e7p+1 + T * (0x1.7bf7d0ba1fd49p-9 + T * (-0x1.618b37483abe8p-21 + T * (0x1.51e0ab53b03a6p-34 + T * -0x1.023798f4a2a00p-48)))) + 0x1.01f60d4fdf3b6p+14)), f[13], tmp);
      tmp = fma(-(0x1.14e7994e1a3f4p+8 * (T * (0x1.c2bc95c7fddb1p+0 + T * (0x1.2d77335291c21p-8 + T * (-0x1.8bb9fb006a417p-20 + T * (0x1.14a3f4fe94722p-32 + T * -0x1.3e714b400a419p-46)))) + -0x1.b55ea88ce703bp+13)), f[14], tmp);
      tmp = fma(-(0x1.2863e90ff9724p+9 * (T * (0x1.256183d389aa6p+1 + T * (0x1.3120cfa66c760p-9 + T * (-0x1.680c0911ecdbfp-21 + T * (0x1.cb7e14e4de1f4p-34 + T * -0x1.e9953783e1eedp-48)))) + 0x1.8ddbffd8adabap+15)), f[15], tmp);
      tmp = fma(-(0x1.79d6b356da017p+7 * (T * (0x1.edc1423f95973p+1 + T * (0x1.214cd7e62db66p-9 + T * (-0x1.8c5b3dc67eba3p-21 + T * (0x1.1fcab1b9912a3p-33 + T * -0x1.542c2854e86a3p-47)))) + -0x1.7cee54fdf3b64p+15)), f[16], tmp);
      tmp = fma(-(0x1.3f5713ad5bee4p+8 * (T * (0x1.0971c7ee6bae0p+2 + T * (0x1.86b42b3f9ab1ep-9 + T * (-0x1.a8a7da8ef5fe7p-21 + T * (0x1.00f66a44e90d0p-33 + T * -0x1.044c229f7f34fp-47)))) + 0x1.953fff2e48e8ap+14)), f[17], tmp);
      tmp = fma(-(0x1.33700096feb4ap+8 * (T * (0x1.8224031487768p+1 + T * (0x1.52803e497ede9p-8 + T * (-0x1.a2d53f48cbb22p-20 + T * (0x1.17b98c3c9686ep-32 + T * -0x1.36c974de2fce9p-46)))) + 0x1.0e69bf6fd21ffp+15)), f[18], tmp);
      tmp = fma(-(0x1.2863e90ff9724p+8 * (T * (0x1.049f4a5d9c3d6p+1 + T * (0x1.dfe6a5720731ep-8 + T * (-0x1.2c3c3485b62c8p-19 + T * (0x1.94aeec15226e0p-32 + T * -0x1.c4e760753f615p-46)))) + 0x1.34be2da122fadp+12)), f[19], tmp);
      tmp = fma(-(0x1.03249374bc6a8p+9 * (T * (0x1.a73c320a693a8p+0 + T * (0x1.488ac88f5e28fp-8 + T * (-0x1.28c3f4ace66e9p-20 + T * (0x1.26ef4a27b854fp-33 + T * -0x1.c5869c71e7825p-48)))) + -0x1.38ccbfb15b574p+13)), f[20], tmp);
      tmp = fma(-(0x1.1e1c0389f83bep+8 * (T * (0x1.f4645cf6d1024p+0 + T * (0x1.1d0972c8defc6p-7 + T * (-0x1.651c92fac6c2cp-19 + T * (0x1.e1a27ccaa5e06p-32 + T * -0x1.0d91ff12db09fp-45)))) + 0x1.91cc28f5c28f6p+13)), f[21], tmp);
      tmp = fma(-(0x1.8b94f63800219p+7 * (T * (0x1.20b91864fbad3p+2 + T * (0x1.2707a6468c0fap-8 + T * (-0x1.75123eb3ba5c4p-20 + T * (0x1.fb9d6149efe38p-33 + T * -0x1.1e5ee25ffae6bp-46)))) + -0x1.d7f0d989df117p+12)), f[22], tmp);
      tmp = fma(-(0x1.954cff43419e3p+7 * (T * (0x1.683486198a14cp+2 + T * (0x1.0bbca21f5e9bfp-9 + T * (-0x1.1d28ea5e6fd95p-21 + T * (0x1.3abf2c56d8d5fp-34 + T * -0x1.17b2431182340p-48)))) + 0x1.2dfcdc28f5c29p+14)), f[23], tmp);
      tmp = fma(-(0x1.0be922424a277p+8 * (T * (0x1.d8a944f2ce3e4p+1 + T * (0x1.1b4df55c881e2p-8 + T * (-0x1.4fa2825a8a1ddp-20 + T * (0x1.b0c96ce8203e2p-33 + T * -0x1.d3552229febefp-47)))) + -0x1.9550335d249e4p+11)), f[24], tmp);
      tmp = fma(-(0x1.4c3397bb73083p+8 * (T * (0x1.957aaf1dba502p+1 + T * (0x1.377101463a6fcp-9 + T * (-0x1.48e6585748e57p-21 + T * (0x1.4e75f1b05c789p-34 + T * -0x1.fed6b3b564915p-49)))) + 0x1.063110a3d70a4p+16)), f[25], tmp);
      tmp = fma(-(0x1.a9c96fa82e87dp+7 * (T * (0x1.898bb8a5a3682p+2 + T * (0x1.3212e5c078a87p-8 + T * (-0x1.4f98067d615fbp-20 + T * (0x1.7b6addd20d988p-33 + T * -0x1.4c0f350fb41cep-47)))) + 0x1.2be2f837b4a23p+15)), f[26], tmp);
      tmp = fma(-(0x1.45a4d67fd3f5bp+7 * (T * (0x1.d0361814f4aecp+2 + T * (0x1.87d7af23d086fp-8 + T * (-0x1.d74c15e1e11bcp-20 + T * (0x1.2e50dd496714ap-32 + T * -0x1.3e80275a3beafp-46)))) + 0x1.eb6383c9eecc0p+15)), f[27], tmp);
      tmp = fma(-(0x1.81f10d173fb7ap+7 * (T * (0x1.02071e6cd2913p+3 + T * (0x1.01f6d02b7c04bp-7 + T * (-0x1.cfb66c12b2299p-20 + T * (0x1.9b10de3c923b6p-33 + T * -0x1.15bd89437d9bcp-47)))) + 0x1.4c1def9db22d1p+12)), f[28], tmp);
      tmp = fma(-(0x1.148494a2b9d3dp+8 * (T * (0x1.1266d373affb0p+0 + T * (0x1.634a9b006255bp-7 + T * (-0x1.c089bdb6616a1p-19 + T * (0x1.304e6c1f3af79p-31 + T * -0x1.56475dfc0f594p-45)))) + -0x1.651325460aa65p+13)), f[29], tmp);
      tmp = fma(-(0x1.9f12d9cf13cefp+7 * (T * (0x1.6844fda07f3bfp+1 + T * (0x1.2ff69d12bb67ap-7 + T * (-0x1.ab4590f77d4a5p-19 + T * (0x1.49c96202a850fp-31 + T * -0x1.abd0be7220bddp-45)))) + 0x1.43744ef34d6a1p+14)), f[30], tmp);
      tmp = fma(-(0x1.a9c96fa82e87dp+6 * (T * (-0x1.a6617a5d2d1b8p-3 + T * (0x1.7c3587c3a5a91p-6 + T * (-0x1.368cdb6dd343cp-17 + T * (0x1.0f114dfad39a2p-29 + T * -0x1.83795c6af5869p-43)))) + 0x1.fa2d6cbfb15b5p+12)), f[31], tmp);
      tmp = fma(-(0x1.af5a836eb4e98p+6 * (T * (0x1.615262ce5664cp+0 + T * (0x1.4afba742defeap-6 + T * (-0x1.0ef3f9a8e695ap-17 + T * (0x1.d9497cdf85b0dp-30 + T * -0x1.5233e2b2fd884p-43)))) + 0x1.2e52b43958106p+15)), f[32], tmp);
      tmp = fma(-(0x1.fef1b93037d63p+6 * (T * (0x1.0dbccff4ca6cdp+2 + T * (0x1.bd5fbfaabbb01p-7 + T * (-0x1.29e746ebfcc91p-18 + T * (0x1.a8a8b6f535c06p-31 + T * -0x1.f49578f685fa6p-45)))) + 0x1.c37cf765fd8aep+14)), f[33], tmp);
      tmp = fma(-(0x1.8b2fe175d13d7p+7 * (T * (0x1.e304cbb91de5cp-2 + T * (0x1.da56952f74035p-7 + T * (-0x1.5e4ff57107a43p-18 + T * (0x1.1abdda6c0ae52p-30 + T * -0x1.7d127c51e6664p-44)))) + 0x1.19822aed13943p+10)), f[34], tmp);
      tmp = fma(-(0x1.4c3397bb73083p+7 * (T * (0x1.3844cbbc5687fp+3 + T * (0x1.f098c1f4d6d2fp-10 + T * (0x1.b64a3c164155ep-24 + T * (-0x1.5c5b043d5fc7cp-33 + T * 0x1.96df91e6bc3dap-46)))) + 0x1.985bbd3c36113p+15)), f[35], tmp);
      tmp = fma(-(0x1.b51158b827fa2p+6 * (T * (0x1.7e3b62413db7fp+1 + T * (0x1.1497c9b930b39p-6 + T * (-0x1.bfecfa8cb0043p-18 + T * (0x1.837a30695a9b9p-30 + T * -0x1.12b8b08e03e9fp-43)))) + 0x1.902e43a29c77ap+15)), f[36], tmp);
      tmp = fma(-(0x1.037d9b6c01b0ep+6 * (T * (0x1.c4acde19fc2a9p+0 + T * (0x1.1a45ef20d54fbp-5 + T * (-0x1.cf6958ad5a986p-17 + T * (0x1.952685dbd1910p-29 + T * -0x1.219328954ba8ep-42)))) + 0x1.c66a3c6a7ef9ep+13)), f[37], tmp);
      tmp = fma(-(0x1.1e523e4e19688p+6 * (T * (0x1.2793bc5fed258p+0 + T * (0x1.0bf86109b70c4p-5 + T * (-0x1.b70270ae35233p-17 + T * (0x1.7f58fd7e1e6f8p-29 + T * -0x1.11cd67a7dc14fp-42)))) + 0x1.06c271758e219p+14)), f[38], tmp);
      tmp = fma(-(0x1.427612472a610p+6 * (T * (0x1.7ebfa91811c4ap+2 + T * (0x1.808ef8f5ad684p-6 + T * (-0x1.2b0ec96978d84p-17 + T * (0x1.f57fe5207cc87p-30 + T * -0x1.5b44f94013013p-43)))) + 0x1.522cd59b3d07dp+15)), f[39], tmp);
      tmp = fma(-(0x1.6cf5cd62f4c1ep+6 * (T * (0x1.a676af33dfab7p+1 + T * (0x1.8942e6d1d3136p-6 + T * (-0x1.376ee95d63b4ep-17 + T * (0x1.096280c15fae5p-29 + T * -0x1.748461054401ep-43)))) + 0x1.53d76dc5d6388p+14)), f[40], tmp);
      tmp = fma(-(0x1.48e3d91c66681p+6 * (T * (0x1.cf3d5e900342dp+2 + T * (0x1.3a6b3ba55718fp-6 + T * (-0x1.e98f907a99010p-18 + T * (0x1.9a5db7bd5ee14p-30 + T * -0x1.1be2937130a6dp-43)))) + 0x1.fb71a083126e9p+15)), f[41], tmp);
      tmp = fma(-(0x1.058c366871d96p+6 * (T * (0x1.9d4d598f935b6p+1 + T * (0x1.0290e103fe76cp-5 + T * (-0x1.a9ac979f543dap-17 + T * (0x1.74a5353114dedp-29 + T * -0x1.0a7bd04156d53p-42)))) + 0x1.75c02b020c49cp+15)), f[42], tmp);
      tmp = fma(-(0x1.45a4d67fd3f5bp+6 * (T * (0x1.742c5116c8ef4p+2 + T * (0x1.6929c14ed23bap-6 + T * (-0x1.19eadf2fe6e2ep-17 + T * (0x1.da5a809896006p-30 + T * -0x1.49623f5160f77p-43)))) + 0x1.0206619652bd4p+15)), f[43], tmp);
      tmp = fma(-(0x1.20d3e75f1f4a5p+6 * (T * (0x1.d3f701135069dp+1 + T * (0x1.d6e2125269b99p-6 + T * (-0x1.7f7e88c4a6b7ep-17 + T * (0x1.4d62a007cdc3ep-29 + T * -0x1.da9e42bc75851p-43)))) + 0x1.df7161ff2e48fp+14)), f[44], tmp);
    } else {
      tmp = fma(-(0x1.28ba9057d1783p+8 * (T * (0x1.a63b0c4588a05p+1 + T * (0x1.712969da04050p-11 + T * (-0x1.629f839620fc6p-20 + T * (0x1.83ae94da0fe59p-30 + T * -0x1.13441e6a0b3dfp-41)))) + -0x1.fe732fec56d5dp+9)), f[0], tmp);
      tmp = fma(-(0x1.01c2d34acaff7p+13 * (T * (0x1.4000000000000p+1 + T * (0x1.8d112bf5fb7e0p-42 + T * (-0x1.7f85eab504006p-51 + T * (0x1.538a620b2373fp-61 + T * -0x1.c09fb31fd8141p-73)))) + 0x1.8e06a3bcd35a8p+14)), f[1], tmp);
      tmp = fma(-(0x1.01c2d350092cdp+12 * (T * (0x1.2c130ac9b2911p+1 + T * (0x1.058175caab342p-8 + T * (-0x1.b3b80759749d1p-18 + T * (0x1.5a4c582f87e3dp-28 + T * -0x1.9f3d0eb996c74p-40)))) + -0x1.caf7b3bfb58d1p+9)), f[2], tmp);
      tmp = fma(-(0x1.03d2b851eb852p+9 * (T * (0x1.9589c6bdbf12dp+1 + T * (-0x1.add3ae5787a18p-10 + T * (0x1.2934a57c4d958p-19 + T * (-0x1.a51e14d5c0503p-30 + T * 0x1.dbba8a635ed80p-42)))) + 0x1.c709096bb98c8p+14)), f[3], tmp);
      tmp = fma(-(0x1.e8d949731098dp+8 * (T * (0x1.080501d23d242p+2 + T * (-0x1.a6c41f6034cc8p-10 + T * (0x1.240abf1dbdb41p-19 + T * (-0x1.8e78ee8cec246p-30 + T * 0x1.d067c130d5fbcp-42)))) + 0x1.a6b138476f2a6p+11)), f[4], tmp);
      tmp = fma(-(0x1.cd7f5ff609dd0p+8 * (T * (0x1.0cb686e536fbfp+2 + T * (-0x1.0aeb63b84c925p-10 + T * (0x1.23b7c52ad124bp-19 + T * (-0x1.7921668781cadp-30 + T * 0x1.8f03963eb52f4p-42)))) + -0x1.d956e8240b780p+14)), f[5], tmp);
      tmp = fma(-(0x1.e8d94983d7907p+7 * (T * (0x1.11abd48f63e0ap+2 + T * (-0x1.1c986431acf9ep-12 + T * (0x1.7652d932e9587p-18 + T * (-0x1.72b101cd97284p-28 + T * 0x1.e584c5e48fadep-40)))) + -0x1.149a541205bc0p+14)), f[6], tmp);
      tmp = fma(-(0x1.03d2b851eb852p+8 * (T * (0x1.e42787ae5fa45p+1 + T * (-0x1.88c9b66c8c0dfp-10 + T * (0x1.b88f92cda255fp-19 + T * (-0x1.4ca5927516966p-29 + T * 0x1.6d361ad59bca4p-41)))) + -0x1.09fc63497b741p+10)), f[7], tmp);
      tmp = fma(-(0x1.f7c6fae7924afp+7 * (T * (0x1.1350a899bcaa1p+2 + T * (-0x1.373d053b75995p-9 + T * (0x1.d94d8bd675c95p-18 + T * (-0x1.a110b0905e0fcp-28 + T * 0x1.058dba115721ap-39)))) + 0x1.26cedbb59ddc2p+8)), f[8], tmp);
      tmp = fma(-(0x1.3f5713b5bf6a1p+9 * (T * (0x1.beb24fde64a4cp+1 + T * (0x1.5390f0fea885dp-13 + T * (-0x1.2e41b3d0faa66p-21 + T * (0x1.b29b14b3f0b25p-31 + T * -0x1.3c9f9bc981c95p-42)))) + 0x1.148d4b1c432cap+16)), f[9], tmp);
      tmp = fma(-(0x1.28d5af07bfe7ep+8 * (T * (0x1.ca2e271a4b2fdp+1 + T * (-0x1.400048c1ba1b0p-12 + T * (0x1.6bee992797344p-22 + T * (0x1.f2a1bae3bf93ap-33 + T * -0x1.97510ba823483p-43)))) + -0x1.c040b020c49bap+13)), f[10], tmp);
      tmp = fma(-(0x1.1e860685553efp+8 * (T * (0x1.0e27e8a748d9cp+2 + T * (-0x1.a9301251f436fp-10 + T * (0x1.34408c703b59dp-18 + T * (-0x1.c97ac86d1539dp-29 + T * 0x1.e8615cf58dbadp-41)))) + 0x1.dff21426fe719p+11)), f[11], tmp);
      tmp = fma(-(0x1.2863e90ff9724p+9 * (T * (0x1.e19f746480de1p+1 + T * (0x1.fbf7d1614006ep-12 + T * (0x1.f42aa330dfb56p-21 + T * (-0x1.08a1f3bd94cffp-30 + T * 0x1.7bf8fa708a0d3p-42)))) + 0x1.67681487fcb92p+15)), f[12], tmp);
      tmp = fma(-(0x1.148494a2b9d3dp+9 * (T * (0x1.d41e76e38c2bfp+1 + T * (0x1.16bcc8dd4edc2p-10 + T * (0x1.e868878cfc8aap-20 + T * (-0x1.c6cad9f474e37p-30 + T * 0x1.159d2d58edf15p-41)))) + 0x1.009add2f1a9fcp+14)), f[13], tmp);
      tmp = fma(-(0x1.14e7994e1a3f4p+8 * (T * (0x1.32cc5c2ed4ffap+2 + T * (-0x1.44ad208e85b45p-8 + T * (0x1.a17083d3e2933p-17 + T * (-0x1.45cdb5fd758e7p-27 + T * 0x1.72e833dfa2eeep-39)))) + -0x1.bf27a7525460bp+13)), f[14], tmp);
      tmp = fma(-(0x1.2863e90ff9724p+9 * (T * (0x1.0cb5ee035346ap+2 + T * (-0x1.3632652eb8373p-10 + T * (0x1.7056246c81ae3p-19 + T * (-0x1.cb9b59fbaac26p-30 + T * 0x1.b58ed1c91768bp-42)))) + 0x1.8a81a1f212d77p+15)), f[15], tmp);
      tmp = fma(-(0x1.79d6b356da017p+7 * (T * (0x1.2daac1343d496p+1 + T * (0x1.266842ab3e914p-8 + T * (-0x1.3eb3eab83633cp-19 + T * (0x1.51fd10511d1a8p-31 + T * -0x1.02ddb83a1a924p-45)))) + -0x1.79e7f07c84b5ep+15)), f[16], tmp);
      tmp = fma(-(0x1.3f5713ad5bee4p+8 * (T * (0x1.9e0b72c73f3bap-1 + T * (0x1.7ec17f4461617p-7 + T * (-0x1.8d40c15d06efbp-17 + T * (0x1.e14c583fde46ap-28 + T * -0x1.de8c6d3a443e1p-40)))) + 0x1.9cf3ec3c9eeccp+14)), f[17], tmp);
      tmp = fma(-(0x1.33700096feb4ap+8 * (T * (0x1.9b3219c31fa4ep+1 + T * (0x1.8d17f1df63fcdp-11 + T * (0x1.21ebbad3d9599p-17 + T * (-0x1.3339cad1d6b94p-27 + T * 0x1.9e3160f1cd550p-39)))) + 0x1.1057b18fc5048p+15)), f[18], tmp);
      tmp = fma(-(0x1.2863e90ff9724p+8 * (T * (0x1.fac71d356ff96p+1 + T * (-0x1.f0244a77197f7p-9 + T * (0x1.3f52277a0a8b7p-16 + T * (-0x1.2908fcc94804cp-26 + T * 0x1.7bd417ca8706cp-38)))) + 0x1.3e1c6a35935fcp+12)), f[19], tmp);
      tmp = fma(-(0x1.03249374bc6a8p+9 * (T * (0x1.498b184c7d064p+2 + T * (-0x1.bfaed90747e6dp-8 + T * (0x1.12d748b9a4c89p-16 + T * (-0x1.9ff6fd8c8b66ap-27 + T * 0x1.d4f26e61176cdp-39)))) + -0x1.4034c95182a99p+13)), f[20], tmp);
      tmp = fma(-(0x1.1e1c0389f83bep+8 * (T * (0x1.139d223a3c91dp+2 + T * (-0x1.125f4e7e42173p-9 + T * (0x1.1605bc90bd661p-16 + T * (-0x1.0152aab0d5df8p-26 + T * 0x1.44699f0472426p-38)))) + 0x1.914d03126e979p+13)), f[21], tmp);
      tmp = fma(-(0x1.8b94f63800219p+7 * (T * (0x1.116315790e08dp+1 + T * (0x1.28dc0ec708b6bp-7 + T * (-0x1.851d295b513c4p-18 + T * (0x1.410e7ab1ff68dp-29 + T * -0x1.c5a468865bde0p-42)))) + -0x1.b82eb04ab606bp+12)), f[22], tmp);
      tmp = fma(-(0x1.954cff43419e3p+7 * (T * (0x1.203868265a06ep+1 + T * (0x1.2142867388492p-7 + T * (-0x1.0967cef8599c0p-17 + T * (0x1.28cb9772e0568p-28 + T * -0x1.1d37b00a8be7dp-40)))) + 0x1.396dcbc6a7efap+14)), f[23], tmp);
      tmp = fma(-(0x1.0be922424a277p+8 * (T * (0x1.ee93ebafbbefep+1 + T * (0x1.6ec96e6bebfdfp-9 + T * (0x1.096ce0e64d114p-19 + T * (-0x1.672b5483bb261p-29 + T * 0x1.ebfb3e2ef3b1bp-41)))) + -0x1.8f3d3cc8de2acp+11)), f[24], tmp);
      tmp = fma(-(0x1.4c3397bb73083p+8 * (T * (0x1.71e04a987f933p+1 + T * (0x1.b76ae82ebca6cp-8 + T * (-0x1.3e82612c20167p-17 + T * (0x1.fa7279086a4c4p-28 + T * -0x1.33bda806adcefp-39)))) + 0x1.051764a8c154dp+16)), f[25], tmp);
      tmp = fma(-(0x1.a9c96fa82e87dp+7 * (T * (0x1.672a8234a31fdp+0 + T * (0x1.ee6ce85d376ddp-7 + T * (-0x1.bda877fc77e6bp-17 + T * (0x1.f849e51f41f92p-28 + T * -0x1.ea1423143389ep-40)))) + 0x1.331da4dd2f1aap+15)), f[26], tmp);
      tmp = fma(-(0x1.45a4d67fd3f5bp+7 * (T * (-0x1.22f59a4800a4ep-5 + T * (0x1.60ac2d35915e1p-6 + T * (-0x1.41f8986c2a345p-16 + T * (0x1.653dab6dde24ep-27 + T * -0x1.53e2298ebef05p-39)))) + 0x1.f6bd518fc5048p+15)), f[27], tmp);
      tmp = fma(-(0x1.81f10d173fb7ap+7 * (T * (0x1.b69ad42c3c9efp+0 + T * (0x1.a0950b6a6c5a7p-7 + T * (0x1.1ae5884a7f06fp-21 + T * (-0x1.38e5016099350p-28 + T * 0x1.f0f4b56ce60d3p-40)))) + 0x1.d6fcf1a9fbe77p+12)), f[28], tmp);
      tmp = fma(-(0x1.148494a2b9d3dp+8 * (T * (0x1.12a6b4b528ec3p+2 + T * (-0x1.688c91f95b2dfp-9 + T * (0x1.4f3aeda131122p-16 + T * (-0x1.3048b1143400cp-26 + T * 0x1.7a244044f8d16p-38)))) + -0x1.6811a4dd2f1aap+13)), f[29], tmp);
      tmp = fma(-(0x1.9f12d9cf13cefp+7 * (T * (0x1.763575adac203p+0 + T * (0x1.9317093d07cbcp-7 + T * (-0x1.a9837a37ac08dp-18 + T * (0x1.279e5de379b7fp-29 + T * -0x1.7770dcf585cb3p-42)))) + 0x1.46e3eacd9e83ep+14)), f[30], tmp);
      tmp = fma(-(0x1.a9c96fa82e87dp+6 * (T * (-0x1.60ff53bd6c5cap+2 + T * (0x1.0860ad1ad40c7p-5 + T * (-0x1.edb368b7d29c0p-17 + T * (0x1.00e9750699a54p-29 + T * 0x1.5d58c552134c5p-41)))) + 0x1.1cb2843d46b27p+13)), f[31], tmp);
      tmp = fma(-(0x1.af5a836eb4e98p+6 * (T * (-0x1.38195eab8701ep+2 + T * (0x1.00bd599769f74p-5 + T * (-0x1.10933abb66c9cp-16 + T * (0x1.e4e479e98cfdep-29 + T * 0x1.d30a2e9946373p-44)))) + 0x1.37ede339c0ebfp+15)), f[32], tmp);
      tmp = fma(-(0x1.fef1b93037d63p+6 * (T * (-0x1.d8385e2ad89bcp+2 + T * (0x1.8e4aac1b8863fp-5 + T * (-0x1.da2d79a880aaap-15 + T * (0x1.460731e83d0a9p-25 + T * -0x1.68575150a0e30p-37)))) + 0x1.dd5ddd6388659p+14)), f[33], tmp);
      tmp = fma(-(0x1.8b2fe175d13d7p+7 * (T * (-0x1.2c7f737f5dec1p-9 + T * (0x1.fc54ec4ad4552p-7 + T * (-0x1.75e964192576fp-18 + T * (0x1.049384aad25cbp-31 + T * 0x1.1961556c85ae7p-42)))) + 0x1.1b97f0995aaf8p+10)), f[34], tmp);
      tmp = fma(-(0x1.4c3397bb73083p+7 * (T * (0x1.62f85428e5ec2p-3 + T * (0x1.73e002f9486fap-6 + T * (-0x1.9850995c2be75p-16 + T * (0x1.ff513db49caa2p-27 + T * -0x1.07dc7cde71947p-38)))) + 0x1.a79fe083126e9p+15)), f[35], tmp);
      tmp = fma(-(0x1.b51158b827fa2p+6 * (T * (-0x1.bb2c88b499fb1p+1 + T * (0x1.d63c00441a21ap-6 + T * (-0x1.13b264336ede7p-16 + T * (0x1.479629c83930cp-28 + T * -0x1.b812222f3d8b7p-42)))) + 0x1.9a54b9096bb99p+15)), f[36], tmp);
      tmp = fma(-(0x1.037d9b6c01b0ep+6 * (T * (-0x1.172dd75917c95p+3 + T * (0x1.af9ec0c249de6p-5 + T * (-0x1.c0595f8fee280p-16 + T * (0x1.7775892d3f086p-28 + T * 0x1.3fe7d29413595p-42)))) + 0x1.044b9096bb98cp+14)), f[37], tmp);
      tmp = fma(-(0x1.1e523e4e19688p+6 * (T * (-0x1.03fbb9a4a6e8ep+3 + T * (0x1.9072c60846fd4p-5 + T * (-0x1.987d498f02598p-16 + T * (0x1.437d056bfaa1ep-28 + T * 0x1.9e67eca672b58p-42)))) + 0x1.238bff9724745p+14)), f[38], tmp);
      tmp = fma(-(0x1.427612472a610p+6 * (T * (-0x1.93d68de0feb30p+2 + T * (0x1.857de9b22d30bp-5 + T * (-0x1.0b3b9f865bcb8p-15 + T * (0x1.aac13c7f0d16fp-27 + T * -0x1.1e84ff1db9db6p-39)))) + 0x1.6549dc0ebedfap+15)), f[39], tmp);
      tmp = fma(-(0x1.6cf5cd62f4c1ep+6 * (T * (-0x1.848391dade5d7p+2 + T * (0x1.561939c3e347ap-5 + T * (-0x1.9ec9eb84f50c7p-16 + T * (0x1.0cff425e97307p-27 + T * -0x1.dd02d04b3ef73p-41)))) + 0x1.7095e28240b78p+14)), f[40], tmp);
      tmp = fma(-(0x1.48e3d91c66681p+6 * (T * (-0x1.1b5d695ce5df1p+2 + T * (0x1.56b310e5b5b9dp-5 + T * (-0x1.e6994769fdcffp-16 + T * (0x1.93f8e90a071dfp-27 + T * -0x1.1e96dea582277p-39)))) + 0x1.07023c63f1412p+16)), f[41], tmp);
      tmp = fma(-(0x1.058c366871d96p+6 * (T * (-0x1.00dea94dec9cfp+3 + T * (0x1.a5942dec43d7fp-5 + T * (-0x1.d28f08862b89ep-16 + T * (0x1.d38668426482ep-28 + T * -0x1.4650077bccc71p-43)))) + 0x1.87b0ab367a0f9p+15)), f[42], tmp);
      tmp = fma(-(0x1.45a4d67fd3f5bp+6 * (T * (-0x1.4d76b09635611p+2 + T * (0x1.6287b313f364dp-5 + T * (-0x1.d88ffbc5422d2p-16 + T * (0x1.6a6d58110178fp-27 + T * -0x1.cbcc68d3e03ebp-40)))) + 0x1.1361b95810625p+15)), f[43], tmp);
      tmp = fma(-(0x1.20d3e75f1f4a5p+6 * (T * (-0x1.17944e81176cbp+3 + T * (0x1.a79d720519df1p-5 + T * (-0x1.023538a6aba05p-15 + T * (0x1.42a85cabc7268p-27 + T * -0x1.f013d29ce5199p-41)))) + 0x1.031833a92a305p+15)), f[44], tmp);
    }
    f[45] = tmp / cpm;
  }
};

}  // namespace tgr
