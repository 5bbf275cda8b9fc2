// mfm_device.hpp -- device-side physics of the multi-fluid MHD patch update.
//
// Per-cell / per-face functions for gfx950.  TF is the arithmetic type of
// reconstruction and Riemann fluxes (double in the parity build, float in the
// fast build); cons->prim recovery, floors, sources and the state update are
// always FP64.  Paths below are relative to MHDAM-3.2.4/ of the reference.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

#include "../../include/mfm.h"

namespace mfm {

// srcIdeal/EosCommon.fh:13-37
constexpr double k1_4PI = 0.079577471545947667884441881686257181;
constexpr double k1_8PI = 0.039788735772973833942220940843128591;
constexpr double kSQRT_2 = 0.707106781186547524400844362104849039;  // 1/sqrt(2)
constexpr double kPI = 3.14159265358979323846264338327950288;
constexpr double k2PI = 6.28318530717958647692528676655900576;
constexpr double k4PI = 12.566370614359172953850573533118;
constexpr double kPI_2 = 1.57079632679489661923132169163975144;
constexpr double kAU = 1.5e13;
constexpr double kNet2Dens = 1.0e-6, kNet2Pres = 1.0e-8;
constexpr double kNet3Dens = 1.0e-7, kNet3Pres = 1.0e-9;

constexpr int kMaxComp = 24;  // 8 + psi + 3*5

// Compile-time equation system: NF fluids (plasma + NF-1 neutrals), DED = 1
// adds the GLM psi component.  Every kernel is instantiated per system so
// all component loops unroll and per-cell vectors live in registers.
template <int NF_, int DED_>
struct Sys {
  static constexpr int NF = NF_;
  static constexpr int DED = DED_;
  static constexpr int NC = 8 + DED_ + 5 * (NF_ - 1);
  static constexpr int IRN = 8 + DED_;  // first neutral component
};

// Constants of one context, passed by value to every kernel (replaces the
// /eos/, /RiemSol/, /Dedner/, /chargeexcm/ and problem COMMON blocks).
struct Consts {
  int dims, nf, nc, dedner, iPsi, iRhoN;
  int flux_kind;      // 0 Roe8, 1 Rusanov, 2 Roe7, 3 HLLC (+ the GLM block with psi)
  int iAveraging;
  int eight_wave, divb_method, problem;
  int8_t lim[kMaxComp];
  int plasma_lim;     // limiter shared by every plasma variable (psi incl.), or -1
  int char_rec;       // plasma slopes limited in characteristic variables
  int tvd_mask;       // bit v: CHECKTVD clips the face values of variable v
  double gamma, invgamma, hgamma, invhgamma, smallr, smallp, del2, smallB;
  double ch, cp;
  int dom_lo[3], dom_hi[3], phys[3];  // phys[d]: non-periodic physical dir
  // Riemann problem
  double rpL[8], rpR[8];
  // heliospheric
  double rp_start_x;
  double sun_xc, sun_yc, sun_zc, sun_r0, sun_rho, sun_p, sun_v, sun_b,
      sun_tilt, sun_int_bc_radius, dir_br_n, omega, lism_v_dim, init_r;
  int sun_b_monopolar;
  double lism_ux, lism_uy, lism_uz, lism_p, lism_m, lism_t, lism_bx, lism_by,
      lism_bz, net_rho, net_p, tmlim, reg_safe_z_top, reg_safe_z_bot;
  double ce_scale_vel, ce_sigma, c13493, c0531;
  int ce_on;
  int ce_mf;          // CHARGE_EXCHANGE_MF: neutral k is born where REG == k
  int axisym;         // coord_sys = 1: geometric sources, r-term of div(B)
  double r0_dt_ignore;  // SW/LISM: the dt exclusion radius
  // uniform factors of HELIOREINIT_DEFAULT, formed once on the host
  double sin_tilt, cos_tilt, sun_beta;
};

// Square root of the flux kernels.  FP64: the Goldschmidt iteration from the
// hardware's reciprocal-square-root estimate with two exact-residual
// corrections (P. Markstein, IA-64 and Elementary Functions, 2000, ch. 9),
// which rounds as sqrt does for arguments above 2^-960, whose residuals are
// normal numbers, without sqrt's rescaling of arguments below 2^-767: 17
// instead of 22 instructions.  Below 2^-960 (a speed under 1e-144) the last bit
// may differ.  Zero and infinity are returned as they are.  Orszag-Tang 512 x 512 x 32 with characteristic slopes 4.94 -> 4.81 ms
// per step, the same bits.
template <typename T>
__device__ __forceinline__ T tsqrt(T x) { return sqrt(x); }
template <>
__device__ __forceinline__ double tsqrt<double>(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double r = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, r, g);
  h = __builtin_fma(h, r, h);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  return __builtin_amdgcn_class(x, 0x260) ? x : g;  // +-0, +inf
}
template <typename T>
__device__ __forceinline__ T tmax(T a, T b) { return a > b ? a : b; }
template <typename T>
__device__ __forceinline__ T tmin(T a, T b) { return a < b ? a : b; }
// Fortran MAX(a, b) with b = floor: returns a if a > b else b
template <typename T>
__device__ __forceinline__ T fmaxr(T b, T a) { return a > b ? a : b; }

// In FP32 a rounding error can push a mathematically non-negative radicand
// below zero; the FP64 build keeps the reference arithmetic untouched.
template <typename T>
__device__ __forceinline__ T nonneg(T x) {
  if constexpr (std::is_same<T, float>::value) return x > 0.f ? x : 0.f;
  return x;
}

// A denominator (not negative) shared by several quotients.  FP64: its
// reciprocal once, by Newton-Raphson from the hardware estimate, then three
// instructions per quotient: q = a r, corrected by the exact remainder,
// q - (q b - a) r (P. Markstein, IBM J. Res. Dev. 34 (1990) 111-119), which
// rounds as the division does; with the remainder's sign taken so, a zero
// keeps a division's sign too.  A full FP64 division takes eleven instructions
// with its scaling for extreme exponents, which the densities, sound speeds and
// pressures divided by here (positive, floored) do not need: without it a
// quotient may round to the neighbour where the remainder underflows (|a| below
// 2^-960), and is a NaN where the denominator is zero or infinite, its
// reciprocal no normal number, or the quotient overflows.  FP32: the
// hardware's reciprocal and a multiply, which is what a division is in the
// FP32 build but for its rescaling of denominators above 2^96 (four more
// instructions per quotient, of use only above 2^126, where the reciprocal is
// no normal number).
// Roe's FP64 flux has some 35 quotients over 11 denominators: 162 instead of
// 198 registers (3 wavefronts per SIMD instead of 2), the same bits; per step
// Brio-Wu 800 84 -> 77 us, Orszag-Tang 512^2 with GLM 153 -> 145 us, 512 x 512 x
// 32 with characteristic slopes 5.33 -> 4.96 ms, four-fluid 128^3 3.27 -> 3.09 ms.
template <typename T>
struct Denom;
template <>
struct Denom<float> {
  float r;
  __device__ __forceinline__ explicit Denom(float d) : r(__builtin_amdgcn_rcpf(d)) {}
  __device__ __forceinline__ Denom(float, double inv) : r((float)inv) {}
  __device__ __forceinline__ float operator()(float a) const { return a * r; }
};
template <>
struct Denom<double> {
  double b, r;
  __device__ __forceinline__ explicit Denom(double d) : b(d) {
    double y = __builtin_amdgcn_rcp(d);
    y = __builtin_fma(__builtin_fma(-d, y, 1.0), y, y);
    r = __builtin_fma(__builtin_fma(-d, y, 1.0), y, y);
  }
  // d with its correctly rounded reciprocal formed on the host
  __device__ __forceinline__ Denom(double d, double inv) : b(d), r(inv) {}
  __device__ __forceinline__ double operator()(double a) const {
    const double q = a * r;
    return __builtin_fma(-__builtin_fma(b, q, -a), r, q);
  }
};

// ------------------------------------------------------------ limiters --
// The smaller of two FP32 slopes of one sign, zero where the signs differ: the
// median of the two and zero.  A NaN in b stays one (the median drops it):
// a slope towards a NaN cell stays an error that the time step reports.
// Minmod 6 instead of 10 instructions, van Leer without branches.
__device__ __forceinline__ float minmod32(float a, float b) {
  const float m = __builtin_amdgcn_fmed3f(a, b, 0.f);
  return b != b ? b : m;
}

// src/reconstructionF.ChF: face values of a cell (left = W-, right = W+)
// from its neighbours wl, wr along the sweep direction.
template <typename T>
__device__ __forceinline__ void limit(int lim, T wl, T w0, T wr, T& left,
                                      T& right) {
  const T dWR = wr - w0, dWL = w0 - wl;
  const T z = T(0), h = T(0.5);
  switch (lim) {
    case MFM_LIM_MINMOD: {  // minmod, :126-155
      if constexpr (std::is_same<T, float>::value) {
        const float sl = 0.5f * minmod32(dWR, dWL);
        left = w0 - sl; right = w0 + sl;
      } else {
        T s = copysign(T(1), dWR);
        T m = s * tmax(z, tmin(fabs(dWR), s * dWL));
        T sl = h * m;
        left = w0 - sl; right = w0 + sl;
      }
      return;
    }
    case MFM_LIM_VANLEER: {  // :794-841 (kappa = 1/3)
      const T BT = T((3.0 - 1.0 / 3.0) / (1.0 - 1.0 / 3.0));
      const T SL1 = T(0.25 * (1.0 - 1.0 / 3.0)), SL2 = T(0.25 * (1.0 + 1.0 / 3.0));
      if constexpr (std::is_same<T, float>::value) {
        const float SL = minmod32(dWR, BT * dWL), SR = minmod32(dWL, BT * dWR);
        left = w0 - (SL1 * SL + SL2 * SR);
        right = w0 + (SL1 * SR + SL2 * SL);
      } else {
        if (dWL * dWR <= z) { left = w0; right = w0; return; }
        T SL = tmin(fabs(dWR), fabs(BT * dWL));
        T SR = tmin(fabs(dWL), fabs(BT * dWR));
        T pl = SL1 * SL + SL2 * SR, pr = SL1 * SR + SL2 * SL;
        if (dWR < z) { pl = -pl; pr = -pr; }
        left = w0 - pl; right = w0 + pr;
      }
      return;
    }
    case MFM_LIM_MC: {  // :622-662
      if (dWL * dWR <= z) { left = w0; right = w0; return; }
      T AR = fabs(dWR), AL = fabs(dWL), s;
      if (T(3) * AL <= AR) s = dWL;
      else if (AL <= T(3) * AR) s = T(0.25) * (dWR + dWL);
      else s = dWR;
      left = w0 - s; right = w0 + s;
      return;
    }
    case MFM_LIM_SUPERBEE: {  // :258-300
      if (dWL * dWR <= z) { left = w0; right = w0; return; }
      T AR = fabs(dWR), AL = fabs(dWL), s;
      if (AL <= h * AR) s = dWL;
      else if (AL <= AR) s = h * dWR;
      else if (AL <= AR + AR) s = h * dWL;
      else s = dWR;
      left = w0 - s; right = w0 + s;
      return;
    }
    case MFM_LIM_VANALBADA: {  // :550-589
      if (dWL * dWR <= z) { left = w0; right = w0; return; }
      const T dS = T(1.0e-6), dSS = T(1.0e-6) + T(1.0e-6);
      T s = h * (dWR * dWL + dS) * (dWR + dWL) / (dWR * dWR + dWL * dWL + dSS);
      left = w0 - s; right = w0 + s;
      return;
    }
    case MFM_LIM_HARMONIC: {  // :492-524
      if (dWL * dWR <= z) { left = w0; right = w0; return; }
      T s = dWR / (T(1) + dWR / dWL);
      left = w0 - s; right = w0 + s;
      return;
    }
    case MFM_LIM_HYPERBEE: {  // :430-464
      if (dWL * dWR <= z) { left = w0; right = w0; return; }
      T A = T(1) + tsqrt(dWR / dWL);
      T s = dWR / (A * A);
      s = s + s;
      left = w0 - s; right = w0 + s;
      return;
    }
    case MFM_LIM_KOREN: {  // :883-918
      if (dWL * dWR <= z) { left = w0; right = w0; return; }
      T H = dWL * dWR / (T(2) * (dWL * dWL + dWR * dWR + T(1.0e-10)) - dWL * dWR);
      left = w0 - (dWL + h * dWR) * H;
      right = w0 + (dWR + h * dWL) * H;
      return;
    }
    case MFM_LIM_VENKAT: {  // :950-988
      if (dWL * dWR <= z) { left = w0; right = w0; return; }
      const T dS = T(1.0e-10), dS2 = T(1.0e-10 * 1.0e-10);
      T H = (dWR + dWL) / (T(6) * (dWR * dWR + dWL * dWL + dS2));
      left = w0 - (dWR + T(2) * dWL) * (dWL + dS) * H;
      right = w0 + (dWL + T(2) * dWR) * (dWR + dS) * H;
      return;
    }
    case MFM_LIM_WENO3: {  // :1096-1136
      T BR = dWR * dWR + T(1.0e-6), AR = T(1) / (BR * BR);
      T BL = dWL * dWL + T(1.0e-6), AL = T(1) / (BL * BL);
      T H = AR / (AR + T(2) * AL);
      left = w0 - h * (dWL + H * (dWR - dWL));
      H = AL / (AL + T(2) * AR);
      right = w0 + h * (dWR - H * (dWR - dWL));
      return;
    }
    case MFM_LIM_WENO3YC: {  // :1169-1212
      T BR = dWR * dWR + T(1.0e-6), BL = dWL * dWL + T(1.0e-6);
      T D2P = dWR - dWL;
      D2P = D2P * D2P;
      T AL = T(1) + D2P / BL, AR = T(1) + D2P / BR;
      T H = AR / (AR + T(2) * AL);
      left = w0 - h * (dWL + H * (dWR - dWL));
      H = AL / (AL + T(2) * AR);
      right = w0 + h * (dWR - H * (dWR - dWL));
      return;
    }
    case MFM_LIM_CD:  // :1056-1079 (W- takes the +1 neighbour, as written)
      left = h * (w0 + wr);
      right = h * (w0 + wl);
      return;
    default:
      left = w0; right = w0;
      return;
  }
}

// ----------------------------------------------------------- face frame --
// The frame of a face of direction d: the normal and the two tangential
// directions as velocity component numbers.  Face arithmetic runs in this
// frame (rho, un, ut1, ut2, p, bn, bt1, bt2, then psi); the rotation is the
// choice of the components to load and store, whose addresses are scalar, so
// one body serves the three directions with d taken at run time.
struct Frame {
  int d, n, t1, t2;
  __device__ __forceinline__ explicit Frame(int dir)
      : d(dir), n(1 + dir), t1(dir == 2 ? 1 : dir + 2), t2(dir == 0 ? 3 : dir) {}
  // component number of frame entry q (0..8) of the plasma
  __device__ __forceinline__ int plasma(int q) const {
    return q == 1 ? n : q == 2 ? t1 : q == 3 ? t2
         : q == 5 ? 4 + n : q == 6 ? 4 + t1 : q == 7 ? 4 + t2 : q;
  }
  // offset of frame entry q (0..4) in a neutral fluid's components
  __device__ __forceinline__ int neutral(int q) const {
    return q == 1 ? n : q == 2 ? t1 : q == 3 ? t2 : q;
  }
  // the limiter of plasma entry q (a scalar select between constant-offset
  // loads: a byte load at a run-time offset would not be scalar)
  __device__ __forceinline__ int limiter(const Consts& C, int q) const {
    auto pick = [](int v, int a, int b, int c) { return v == 1 ? a : v == 2 ? b : c; };
    if (q >= 1 && q <= 3)
      return pick(plasma(q), C.lim[1], C.lim[2], C.lim[3]);
    if (q >= 5 && q <= 7)
      return pick(plasma(q) - 4, C.lim[5], C.lim[6], C.lim[7]);
    return C.lim[q];
  }
};

// ----------------------------------------- characteristic reconstruction --
// *FACESLOPES (src/reconstructionF.ChF): limited slopes SL (lo side) and SR
// (hi side) of a cell from its one-sided differences dSL = W - W(i-1),
// dSR = W(i+1) - W, taken in characteristic variables.
template <typename T>
__device__ __forceinline__ void face_slopes(int lim, T dSL, T dSR, T& SL, T& SR) {
  const T z = T(0), h = T(0.5);
  T s = z;
  switch (lim) {
    case MFM_LIM_MINMOD: {  // MINMODFACESLOPES :157-177
      T sg = copysign(T(1), dSR);
      s = h * (sg * tmax(z, tmin(fabs(dSR), sg * dSL)));
      break;
    }
    case MFM_LIM_VANLEER: {  // VANLEERFACESLOPES :843-881 (kappa = 1/3)
      T pl = z, pr = z;
      if (dSL * dSR > z) {
        const T BT = T((3.0 - 1.0 / 3.0) / (1.0 - 1.0 / 3.0));
        const T SL1 = T(0.25 * (1.0 - 1.0 / 3.0)), SL2 = T(0.25 * (1.0 + 1.0 / 3.0));
        T a = tmin(fabs(dSR), fabs(BT * dSL));
        T b = tmin(fabs(dSL), fabs(BT * dSR));
        pl = SL1 * a + SL2 * b;
        pr = SL1 * b + SL2 * a;
        if (dSR < z) { pl = -pl; pr = -pr; }
      }
      SL = pl; SR = pr;
      return;
    }
    case MFM_LIM_MC:  // MCFACESLOPES :664-694
      if (dSL * dSR > z) {
        T AR = fabs(dSR), AL = fabs(dSL);
        if (T(3) * AL <= AR) s = dSL;
        else if (AL <= T(3) * AR) s = T(0.25) * (dSR + dSL);
        else s = dSR;
      }
      break;
    case MFM_LIM_SUPERBEE:  // SUPERBEEFACESLOPES :356-388
      if (dSL * dSR > z) {
        T AR = fabs(dSR), AL = fabs(dSL);
        if (AL <= h * AR) s = dSL;
        else if (AL <= AR) s = h * dSR;
        else if (AL <= AR + AR) s = h * dSL;
        else s = dSR;
      }
      break;
    case MFM_LIM_VANALBADA:  // VANALBADAFACESLOPES :591-620
      if (dSL * dSR > z) {
        const T dS = T(1.0e-6), dSS = T(1.0e-6) + T(1.0e-6);
        s = h * (dSR * dSL + dS) * (dSR + dSL) / (dSR * dSR + dSL * dSL + dSS);
      }
      break;
    case MFM_LIM_HARMONIC:  // HARMONICFACESLOPES :526-548
      if (dSL * dSR > z) s = dSR * dSL / (dSL + dSR);
      break;
    case MFM_LIM_HYPERBEE:  // HYPERBEEFACESLOPES :466-490
      if (dSL * dSR > z) {
        T A = T(1) + tsqrt(dSR / dSL);
        s = dSR / (A * A);
        s = s + s;
      }
      break;
    case MFM_LIM_KOREN: {  // KORENFACESLOPES :920-948
      T pl = z, pr = z;
      if (dSL * dSR > z) {
        T H = dSL * dSR / (T(2) * (dSL * dSL + dSR * dSR + T(1.0e-10)) - dSL * dSR);
        pl = (dSL + h * dSR) * H;
        pr = (dSR + h * dSL) * H;
      }
      SL = pl; SR = pr;
      return;
    }
    case MFM_LIM_VENKAT: {  // VENKATAKRISHNANFACESLOPES :990-1020
      T pl = z, pr = z;
      if (dSL * dSR > z) {
        const T dS = T(1.0e-10), dS2 = T(1.0e-10 * 1.0e-10);
        T H = (dSR + dSL) / (T(6) * (dSR * dSR + dSL * dSL + dS2));
        pl = (dSR + T(2) * dSL) * (dSL + dS) * H;
        pr = (dSL + T(2) * dSR) * (dSR + dS) * H;
      }
      SL = pl; SR = pr;
      return;
    }
    case MFM_LIM_WENO3: {  // WENO3FACESLOPES :1138-1167
      T BR = dSR * dSR + T(1.0e-6), AR = T(1) / (BR * BR);
      T BL = dSL * dSL + T(1.0e-6), AL = T(1) / (BL * BL);
      T H = AR / (AR + T(2) * AL);
      SL = h * (dSL + H * (dSR - dSL));
      H = AL / (AL + T(2) * AR);
      SR = h * (dSR - H * (dSR - dSL));
      return;
    }
    case MFM_LIM_WENO3YC: {  // WENO3YCFACESLOPES :1214-1247
      T BR = dSR * dSR + T(1.0e-6), BL = dSL * dSL + T(1.0e-6);
      T D2P = dSR - dSL;
      D2P = D2P * D2P;
      T AL = T(1) + D2P / BL, AR = T(1) + D2P / BR;
      T H = AR / (AR + T(2) * AL);
      SL = h * (dSL + H * (dSR - dSL));
      H = AL / (AL + T(2) * AR);
      SR = h * (dSR - H * (dSR - dSL));
      return;
    }
    case MFM_LIM_CD:  // CDFACESLOPES :1081-1094
      SL = h * dSL; SR = h * dSR;
      return;
    default:  // no limiter: the slopes stay as they are
      SL = dSL; SR = dSR;
      return;
  }
  SL = s; SR = s;
}

// minmod3 (src/reconstructionF.ChF:16-26)
template <typename T>
__device__ __forceinline__ T minmod3(T A, T B, T C) {
  const T sg = copysign(T(1), A);
  return sg * tmax(T(0), tmin(tmin(fabs(A), sg * B), sg * C));
}

// CHECKTVD (src/reconstructionF.ChF:1248-1278) on one face value: the
// slope W - W- (lo) or W+ - W (hi) is clipped to the cell's one-sided
// differences.
template <typename T>
__device__ __forceinline__ T tvd_lo(T wm, T w0, T dWL, T dWR) {
  return w0 - minmod3(dWL, dWR, w0 - wm);
}
template <typename T>
__device__ __forceinline__ T tvd_hi(T wp, T w0, T dWL, T dWR) {
  return w0 + minmod3(dWL, dWR, wp - w0);
}

// Eigen-structure of the ideal-MHD system at one cell along the normal of
// the face frame, formed from the cell's primitive state as in CHARANALYSISF / CHARSYNTHESISF
// (srcIdeal/PatchIdealMHDF.ChF:1167-1505).  The fast / slow weights take the
// degenerate branch below 1e-12 in the analysis (aF, aS) and below 1e-8 in
// the synthesis (aF2, aS2).
template <typename T>
struct CharBasis {
  T Rho, cc, c, af, as, aF, aS, aF2, aS2, betaY, betaZ, BX;
  // the analysis's denominators: cc, 2 cc, 2 Rho cc, 2 sqrt(2 pi Rho),
  // 4 c sqrt(pi Rho)
  Denom<T> byCc, by2Cc, by2RhoCc, by2Sq, by4cSq;
};

template <typename T>
__device__ __forceinline__ void char_alpha(T dfs, T cc, T aas, T aaf, T eps, T& aF, T& aS) {
  if (dfs < eps) { aF = T(1); aS = T(0); }
  else if ((cc - aas) <= T(0)) { aF = T(0); aS = T(1); }
  else if ((aaf - cc) <= T(0)) { aF = T(1); aS = T(0); }
  else {
    const Denom<T> byDfs(dfs);
    aF = tsqrt(byDfs(cc - aas));
    aS = tsqrt(byDfs(aaf - cc));
  }
}

template <typename T>
__device__ __forceinline__ CharBasis<T> char_basis(const Consts& C, const T* w) {
  constexpr int bn = 5, bt1 = 6, bt2 = 7;
  const T PGas = fmaxr((T)C.smallp, w[4]);
  const T Rho = fmaxr((T)C.smallr, w[0]);
  const T BX = w[bn], BY = w[bt1], BZ = w[bt2];
  const Denom<T> byRho(Rho);
  const T cc = byRho(T(C.gamma) * PGas);
  const T c = tsqrt(cc);
  const T BX2 = BX * BX, BY2 = BY * BY, BZ2 = BZ * BZ;
  const T BYZ2 = BY2 + BZ2;
  const T BxBH = T(k1_8PI) * (BX2 + BYZ2);
  const T bb = byRho(T(k1_4PI) * BX2);
  const T b = tsqrt(bb);
  T aas, as, aaf, af, betaY, betaZ;
  if (BYZ2 < T(C.smallB) * T(C.smallB)) {
    betaY = T(kSQRT_2);
    betaZ = T(kSQRT_2);
    if (bb > cc) { aaf = bb; aas = cc; af = b; as = c; }
    else { aaf = cc; aas = bb; af = c; as = b; }
  } else {
    const T hyz = tsqrt(BYZ2);
    const Denom<T> byHyz(hyz);
    betaY = byHyz(BY);
    betaZ = byHyz(BZ);
    const T szb = cc + byRho(BxBH + BxBH);
    const T h = tsqrt(nonneg(szb * szb - T(4) * cc * bb));
    aas = T(0.5) * (szb - h);
    as = tsqrt(nonneg(aas));
    aaf = T(0.5) * (szb + h);
    af = tsqrt(aaf);
  }
  const T dfs = aaf - aas;
  T aF, aS;
  char_alpha<T>(dfs, cc, aas, aaf, T(1.0e-12), aF, aS);
  // with the wider threshold the weights differ only inside it
  const bool deg = dfs < T(1.0e-8);
  return CharBasis<T>{Rho, cc, c, af, as, aF, aS, deg ? T(1) : aF, deg ? T(0) : aS,
                      betaY, betaZ, BX, Denom<T>(cc), Denom<T>(T(2) * cc),
                      Denom<T>(T(2) * Rho * cc), Denom<T>(T(2) * tsqrt(T(k2PI) * Rho)),
                      Denom<T>(T(4) * c * tsqrt(T(kPI) * Rho))};
}

// CHARANALYSISF (:1252-1325): primitive differences d (plasma components in
// the face frame) -> characteristic variables a (entropy, div(B), two
// Alfven, two fast, two slow).
template <typename T>
__device__ __forceinline__ void char_analysis(const CharBasis<T>& B, const T* d, T* a) {
  constexpr int n = 1, t1 = 2, t2 = 3, bn = 5, bt1 = 6, bt2 = 7;
  // SIGN(one, BX) with -0.0 counted as positive, as the synthesis's BX < 0
  // test does, so that both transforms agree where the field is exactly zero
  const T siBX = B.BX < T(0) ? T(-1) : T(1);
  const T dP = d[4], dRho = d[0], dUn = d[n], dUt1 = d[t1], dUt2 = d[t2];
  const T dBn = d[bn], dBt1 = d[bt1], dBt2 = d[bt2];
  a[0] = dRho - B.byCc(dP);
  a[1] = dBn;
  T h1 = T(kSQRT_2) * (B.betaY * dUt2 - B.betaZ * dUt1);
  T h2 = B.by2Sq(siBX * (B.betaZ * dBt1 - B.betaY * dBt2));
  a[2] = h1 + h2;
  a[3] = h1 - h2;
  h1 = B.by2RhoCc(dP);
  h2 = B.by2Cc(dUn);
  const T h3 = B.by4cSq(B.betaY * dBt1 + B.betaZ * dBt2);
  const T h4 = B.by2Cc(siBX * (B.betaY * dUt1 + B.betaZ * dUt2));
  const T aF = B.aF, aS = B.aS, af = B.af, as = B.as;
  a[4] = aF * (h1 + af * h2) + aS * (h3 - as * h4);
  a[5] = aF * (h1 - af * h2) + aS * (h3 + as * h4);
  a[6] = aS * (h1 + as * h2) - aF * (h3 - af * h4);
  a[7] = aS * (h1 - as * h2) - aF * (h3 + af * h4);
}

// CHARSYNTHESISF (:1438-1502): characteristic variables -> primitive
// differences.
template <typename T>
__device__ __forceinline__ void char_synthesis(const CharBasis<T>& B, const T* a, T* d) {
  constexpr int n = 1, t1 = 2, t2 = 3, bn = 5, bt1 = 6, bt2 = 7;
  const T betaYX = B.BX < T(0) ? -B.betaY : B.betaY;
  const T betaZX = B.BX < T(0) ? -B.betaZ : B.betaZ;
  const T alpha3 = T(kSQRT_2) * a[2], alpha4 = T(kSQRT_2) * a[3];
  const T a3p4 = alpha3 + alpha4, a3m4 = alpha3 - alpha4;
  const T a5p6 = a[4] + a[5], a5m6 = a[4] - a[5];
  const T a7p8 = a[6] + a[7], a7m8 = a[6] - a[7];
  const T DN = T(2) * tsqrt(T(kPI) * B.Rho);
  const T aF = B.aF2, aS = B.aS2;
  const T HRho = B.Rho * (aF * a5p6 + aS * a7p8);
  const T HU = aS * B.as * a5m6 - aF * B.af * a7m8;
  const T HB = B.c * (aS * a5p6 - aF * a7p8);
  d[0] = a[0] + HRho;
  d[n] = aF * B.af * a5m6 + aS * B.as * a7m8;
  d[t1] = -B.betaZ * a3p4 - betaYX * HU;
  d[t2] = B.betaY * a3p4 - betaZX * HU;
  d[4] = B.cc * HRho;
  d[bn] = a[1];
  d[bt1] = DN * (betaZX * a3m4 + B.betaY * HB);
  d[bt2] = DN * (-betaYX * a3m4 + B.betaZ * HB);
}

// ---------------------------------------------------- cons -> prim (FP64) --
// CONSTOPRIM / CONSTOPRIM_MF (srcIdeal/PatchIdealMHDF.ChF:143-189,
// srcIdeal/PatchMHDMFF.ChF:5-80): the multi-fluid version floors rho.
// One neutral fluid (5 components).
__device__ __forceinline__ void neutral_to_prim(const Consts& C, const double* u, double* w) {
  const double r = fmaxr(C.smallr, u[0]);
  const double jr = 1.0 / r;
  const double ax = u[1] * jr, ay = u[2] * jr, az = u[3] * jr;
  const double k2 = u[1] * ax + u[2] * ay + u[3] * az;
  double q = C.hgamma * (u[4] - 0.5 * k2);
  q = fmaxr(C.smallp, q);
  w[0] = r; w[1] = ax; w[2] = ay; w[3] = az; w[4] = q;
}

// The plasma (8 components).
template <class S>
__device__ __forceinline__ void plasma_to_prim(const Consts& C, const double* u, double* w) {
  double rho = u[0];
  if (S::NF > 1) rho = fmaxr(C.smallr, u[0]);
  const double ir = 1.0 / rho;
  const double vx = u[1] * ir, vy = u[2] * ir, vz = u[3] * ir;
  const double ke = u[1] * vx + u[2] * vy + u[3] * vz;
  const double b = k1_4PI * (u[5] * u[5] + u[6] * u[6] + u[7] * u[7]);
  double p = C.hgamma * (u[4] - 0.5 * (ke + b));
  p = fmaxr(C.smallp, p);
  w[0] = rho; w[1] = vx; w[2] = vy; w[3] = vz; w[4] = p;
  w[5] = u[5]; w[6] = u[6]; w[7] = u[7];
}

template <class S>
__device__ __forceinline__ void cons_to_prim(const Consts& C, const double* u,
                                             double* w) {
  plasma_to_prim<S>(C, u, w);
  if (S::DED) w[8] = u[8];
#pragma unroll
  for (int f = 1; f < S::NF; ++f)
    neutral_to_prim(C, u + S::IRN + 5 * (f - 1), w + S::IRN + 5 * (f - 1));
}

// ---------------------------------------------------------- MHD fluxes --
// Rotated plasma state: p, rho, un, ut1, ut2, bn, bt1, bt2.
template <typename T>
struct MState { T p, rho, u, v, w, bx, by, bz; };

// Differences (left - right) of the conserved variables (cons) and the
// primitive-like jumps the left eigenvectors act on (out): the du block of
// RIEMANNF / RIEMANN7F (src/Roe8WaveF.ChF).
template <typename T, bool seven>
__device__ __forceinline__ void roe_jumps(const Consts& C, const MState<T>& L,
                                          const MState<T>& R, const Denom<T>& byRho, T U_, T V_,
                                          T W_, T BX_, T BY_, T BZ_, T kk_, T* out,
                                          T* cons) {
  using D = T;
  const D half = D(0.5), c4 = D(k1_4PI), c8 = D(k1_8PI), hg = D(C.hgamma);
  const D Lr = L.rho, Lu = L.u, Lv = L.v, Lw = L.w, Lp = L.p, Lbx = L.bx, Lby = L.by, Lbz = L.bz;
  const D Rr = R.rho, Ru = R.u, Rv = R.v, Rw = R.w, Rp = R.p, Rbx = R.bx, Rby = R.by, Rbz = R.bz;
  const Denom<T> byHg((T)C.hgamma, C.invhgamma);
  const D U = U_, V = V_, W = W_, BX = BX_, BY = BY_, BZ = BZ_, kk = kk_;
  const D RUL = Lr * Lu, RVL = Lr * Lv, RWL = Lr * Lw;
  const D BxBL = c8 * (Lbx * Lbx + Lby * Lby + Lbz * Lbz);
  const D RUxUL = half * (RUL * Lu + RVL * Lv + RWL * Lw);
  const D EL = byHg(Lp) + RUxUL + BxBL;
  const D RUR = Rr * Ru, RVR = Rr * Rv, RWR = Rr * Rw;
  const D BxBR = c8 * (Rbx * Rbx + Rby * Rby + Rbz * Rbz);
  const D RUxUR = half * (RUR * Ru + RVR * Rv + RWR * Rw);
  const D ER = byHg(Rp) + RUxUR + BxBR;
  D du1 = Lr - Rr, du2 = RUL - RUR, du3 = RVL - RVR, du4 = RWL - RWR;
  D du5 = EL - ER;
  const D du6 = Lbx - Rbx, du7 = Lby - Rby, du8 = Lbz - Rbz;
  cons[0] = T(du1); cons[1] = T(du2); cons[2] = T(du3); cons[3] = T(du4);
  cons[4] = T(du5); cons[5] = T(du6); cons[6] = T(du7); cons[7] = T(du8);
  if constexpr (!seven) {
    du5 = -hg * (-kk * du1 + U * du2 + V * du3 + W * du4 - du5 +
                 (BX * du6 + BY * du7 + BZ * du8) * c4);
  } else {
    du5 = -hg * (-kk * du1 + U * du2 + V * du3 + W * du4 - du5 +
                 (BY * du7 + BZ * du8) * c4);
  }
  du2 = byRho(-U * du1 + du2);
  du3 = byRho(-V * du1 + du3);
  du4 = byRho(-W * du1 + du4);
  out[0] = T(du1); out[1] = T(du2); out[2] = T(du3); out[3] = T(du4);
  out[4] = T(du5); out[5] = T(du6); out[6] = T(du7); out[7] = T(du8);
}

// 8-wave Roe flux (RIEMANNF, src/Roe8WaveF.ChF:5-601), left/right already
// clamped to (smallp, smallr).  Only the non-zero eigenvector entries are
// formed; the sums keep the reference's term order, so the FP64 build is
// bit-compatible with the dense form.  out order: rho, mn, mt1, mt2, E, bn,
// bt1, bt2.  seven = true gives RIEMANN7F (src/Roe7WaveF.ChF:5-558): no B_n
// wave, out[5] = 0.
template <typename T, bool seven>
__device__ __forceinline__ void roe_flux(const Consts& C, const MState<T>& L,
                                         const MState<T>& R, T* out) {
  const T half = T(0.5), one = T(1), zero = T(0), two = T(2);
  const T g = T(C.gamma), hg = T(C.hgamma);
  const T c4 = T(k1_4PI), c8 = T(k1_8PI), rs2 = T(kSQRT_2);
  const Denom<T> byHg(hg, C.invhgamma), byRhoL(L.rho), byRhoR(R.rho);

  const T RUL = L.rho * L.u, RVL = L.rho * L.v, RWL = L.rho * L.w;
  const T BxBL = c8 * (L.bx * L.bx + L.by * L.by + L.bz * L.bz);
  const T RUxUL = half * (RUL * L.u + RVL * L.v + RWL * L.w);
  const T PL = L.p + BxBL;
  const T EL = byHg(L.p) + RUxUL + BxBL;
  const T AL2 = byRhoL(g * L.p);
  const T RUR = R.rho * R.u, RVR = R.rho * R.v, RWR = R.rho * R.w;
  const T BxBR = c8 * (R.bx * R.bx + R.by * R.by + R.bz * R.bz);
  const T RUxUR = half * (RUR * R.u + RVR * R.v + RWR * R.w);
  const T PR = R.p + BxBR;
  const T ER = byHg(R.p) + RUxUR + BxBR;
  const T AR2 = byRhoR(g * R.p);
  T ccmi, ccma;
  if (AL2 > AR2) { ccmi = AR2; ccma = AL2; } else { ccmi = AL2; ccma = AR2; }

  T Rho, U, V, W, BX, BY, BZ, BX2, BYZ2, BxBH, kk, cc;
  if (C.iAveraging == 1) {
    const T HL = byRhoL(EL + PL), HR = byRhoR(ER + PR);
    const T cL = one / (one + tsqrt(byRhoL(R.rho)));
    const T cR = one - cL;
    Rho = R.rho * cL + L.rho * cR;
    U = L.u * cL + R.u * cR;
    V = L.v * cL + R.v * cR;
    W = L.w * cL + R.w * cR;
    const T HAV = HL * cL + HR * cR;
    BX = R.bx * cL + L.bx * cR;
    BY = R.by * cL + L.by * cR;
    BZ = R.bz * cL + L.bz * cR;
    const T BXAV = half * (L.bx + R.bx);
    BX2 = BXAV * BXAV;
    BYZ2 = BY * BY + BZ * BZ;
    BxBH = c8 * (BX2 + BYZ2);
    kk = half * (U * U + V * V + W * W);
    const T dbx = R.bx - L.bx, dby = R.by - L.by, dbz = R.bz - L.bz;
    const T X = byRhoL(c8 * (dbx * dbx + dby * dby + dbz * dbz) * cL * cL);
    cc = hg * (HAV - kk - Denom<T>(Rho)(c4 * (BX * BXAV + BYZ2))) + (two - g) * X;
  } else {
    Rho = half * (L.rho + R.rho);
    U = half * (L.u + R.u); V = half * (L.v + R.v); W = half * (L.w + R.w);
    BX = half * (L.bx + R.bx); BY = half * (L.by + R.by); BZ = half * (L.bz + R.bz);
    const T P = half * (PL + PR);
    BX2 = BX * BX;
    BYZ2 = BY * BY + BZ * BZ;
    BxBH = c8 * (BX2 + BYZ2);
    kk = half * (U * U + V * V + W * W);
    cc = Denom<T>(Rho)(g * (P - BxBH));
  }
  const Denom<T> byRho(Rho);
  const T bb = byRho(c4 * BX2);
  const T b = tsqrt(bb);
  if (cc < ccmi) cc = ccmi;
  if (cc > ccma) cc = ccma;
  const T c = tsqrt(cc);

  T hyy, hzz, aaf, aas, af, as;
  const T sB = T(C.smallB);
  if (BYZ2 < sB * sB) {
    hyy = rs2; hzz = rs2;
    if (bb > cc) { aaf = bb; aas = cc; af = b; as = c; }
    else { aaf = cc; aas = bb; af = c; as = b; }
  } else {
    const T hyz = tsqrt(BYZ2);
    const Denom<T> byHyz(hyz);
    hyy = byHyz(BY); hzz = byHyz(BZ);
    const T szb = cc + byRho(BxBH + BxBH);
    const T hh = tsqrt(nonneg(szb * szb - T(4) * cc * bb));
    aas = half * (szb - hh);
    if (aas <= zero) { aas = zero; as = zero; }
    else if (aas >= cc) { aas = cc; as = c; }
    else as = tsqrt(aas);
    aaf = half * (szb + hh);
    if (aaf <= cc) { aaf = cc; af = c; }
    else af = tsqrt(aaf);
  }

  // |lambda| with the entropy fix
  T A1, A3, A4, A5, A6, A7, A8;  // A2 == A1 (both |U|)
  {
    const T eigmax = fabs(U) + fabs(V) + fabs(W) + af;
    const T del = T(C.del2) * eigmax;
    const T dl2 = del * del;
    const Denom<T> byDel(del);
    auto fix = [&](T e) -> T {
      const T zz = fabs(e);
      return zz >= del ? zz : byDel(half * (zz * zz + dl2));
    };
    A1 = fix(U); A3 = fix(U + b); A4 = fix(U - b);
    A5 = fix(U + af); A6 = fix(U - af); A7 = fix(U + as); A8 = fix(U - as);
  }
  const T dfs = aaf - aas;
  T alf, als;
  if (dfs < T(1.0e-8)) { alf = one; als = zero; }
  else if ((cc - aas) <= zero) { alf = zero; als = one; }
  else if ((aaf - cc) <= zero) { alf = one; als = zero; }
  else {
    const Denom<T> byDfs(dfs);
    alf = tsqrt(byDfs(cc - aas));
    als = tsqrt(byDfs(aaf - cc));
  }
  const T sih = (BX >= zero) ? one : -one;

  T du[8], dcons[8];
  roe_jumps<T, seven>(C, L, R, byRho, U, V, W, BX, BY, BZ, kk, du, dcons);
  const T du1 = du[0], du2 = du[1], du3 = du[2], du4 = du[3], du5 = du[4];
  const T du6 = du[5], du7 = du[6], du8 = du[7];
  const T sqPiRho = tsqrt(T(kPI) * Rho), sq2PiRho = tsqrt(T(k2PI) * Rho);

  // non-zero entries of the left/right eigenvector matrices
  const Denom<T> byCc(cc), bySq2(sq2PiRho), byCcRho(cc * Rho);
  const T ic = byCc(one);
  const T aff = alf * af, ass = als * as;
  const T hzs = hzz * rs2, hys = hyy * rs2;
  const T q7 = bySq2(half * hzz * sih), q8 = bySq2(half * hyy * sih);
  const Denom<T> byCsp(c * sqPiRho);
  // fast/slow rows
  const T so52 = byCc(half * alf * af);
  const T so53 = byCc(-half * als * as * hyy * sih);
  const T so54 = byCc(-half * als * as * hzz * sih);
  const T so55 = byCcRho(half * alf);
  const T so57 = byCsp(T(0.25) * als * hyy), so58 = byCsp(T(0.25) * als * hzz);
  const T so72 = byCc(half * als * as);
  const T so73 = byCc(half * alf * af * hyy * sih);
  const T so74 = byCc(half * alf * af * hzz * sih);
  const T so75 = byCcRho(half * als);
  const T so77 = byCsp(-T(0.25) * alf * hyy), so78 = byCsp(-T(0.25) * alf * hzz);

  const T ra_f = Rho * alf, ra_s = Rho * als;
  const T sp35 = -ass * hyy * sih, sp37 = aff * hyy * sih;
  const T sp45 = -ass * hzz * sih, sp47 = aff * hzz * sih;
  const T sp55 = alf * Rho * cc, sp57 = als * Rho * cc;
  const T sp73 = hzz * sq2PiRho * sih, sp83 = -hyy * sq2PiRho * sih;
  const T sp75 = two * als * sqPiRho * c * hyy, sp77 = -two * alf * sqPiRho * c * hyy;
  const T sp85 = two * als * sqPiRho * c * hzz, sp87 = -two * alf * sqPiRho * c * hzz;

  T ra1, ra2, ra3, ra4, ra5, ra6, ra7, ra8;
  const T so15 = -ic;
  const T lu1 = A1 * (du1 + so15 * du5);
  const T lu3 = A3 * (-hzs * du3 + hys * du4 + q7 * du7 + (-q8) * du8);
  const T lu4 = A4 * (-hzs * du3 + hys * du4 + (-q7) * du7 + q8 * du8);
  const T lu5 = A5 * (so52 * du2 + so53 * du3 + so54 * du4 + so55 * du5 +
                      so57 * du7 + so58 * du8);
  const T lu6 = A6 * ((-so52) * du2 + (-so53) * du3 + (-so54) * du4 +
                      so55 * du5 + so57 * du7 + so58 * du8);
  const T lu7 = A7 * (so72 * du2 + so73 * du3 + so74 * du4 + so75 * du5 +
                      so77 * du7 + so78 * du8);
  const T lu8 = A8 * ((-so72) * du2 + (-so73) * du3 + (-so74) * du4 +
                      so75 * du5 + so77 * du7 + so78 * du8);

  ra1 = lu1 + ra_f * lu5 + ra_f * lu6 + ra_s * lu7 + ra_s * lu8;
  ra2 = aff * lu5 + (-aff) * lu6 + ass * lu7 + (-ass) * lu8;
  ra3 = -hzs * lu3 + (-hzs) * lu4 + sp35 * lu5 + (-sp35) * lu6 + sp37 * lu7 +
          (-sp37) * lu8;
  ra4 = hys * lu3 + hys * lu4 + sp45 * lu5 + (-sp45) * lu6 + sp47 * lu7 +
          (-sp47) * lu8;
  ra5 = sp55 * lu5 + sp55 * lu6 + sp57 * lu7 + sp57 * lu8;
  ra7 = sp73 * lu3 + (-sp73) * lu4 + sp75 * lu5 + sp75 * lu6 + sp77 * lu7 +
          sp77 * lu8;
  ra8 = sp83 * lu3 + (-sp83) * lu4 + sp85 * lu5 + sp85 * lu6 + sp87 * lu7 +
          sp87 * lu8;
  ra6 = zero;
  if constexpr (!seven) {
    ra6 = A1 * du6;  // lu2 = |U| * du6, sp62 = 1
    ra5 = ra1 * kk + Rho * (U * ra2 + V * ra3 + W * ra4) + byHg(ra5) +
          c4 * (BX * ra6 + BY * ra7 + BZ * ra8);
  } else {
    ra5 = ra1 * kk + Rho * (U * ra2 + V * ra3 + W * ra4) + byHg(ra5) +
          c4 * (BY * ra7 + BZ * ra8);
  }

  ra2 = U * ra1 + Rho * ra2;
  ra3 = V * ra1 + Rho * ra3;
  ra4 = W * ra1 + Rho * ra4;

  const T fl1 = RUL, fr1 = RUR;
  const T fl2 = L.u * RUL - L.bx * L.bx * c4 + PL;
  const T fr2 = R.u * RUR - R.bx * R.bx * c4 + PR;
  const T fl3 = L.u * RVL - L.bx * L.by * c4, fr3 = R.u * RVR - R.bx * R.by * c4;
  const T fl4 = L.u * RWL - L.bx * L.bz * c4, fr4 = R.u * RWR - R.bx * R.bz * c4;
  const T fl5 = L.u * (EL + PL) - L.bx * (L.u * L.bx + L.v * L.by + L.w * L.bz) * c4;
  const T fr5 = R.u * (ER + PR) - R.bx * (R.u * R.bx + R.v * R.by + R.w * R.bz) * c4;
  const T fl7 = L.u * L.by - L.bx * L.v, fr7 = R.u * R.by - R.bx * R.v;
  const T fl8 = L.u * L.bz - L.bx * L.w, fr8 = R.u * R.bz - R.bx * R.w;
  out[0] = half * (fl1 + fr1 + ra1);
  out[1] = half * (fl2 + fr2 + ra2);
  out[2] = half * (fl3 + fr3 + ra3);
  out[3] = half * (fl4 + fr4 + ra4);
  out[4] = half * (fl5 + fr5 + ra5);
  out[5] = seven ? zero : half * (zero + zero + ra6);
  out[6] = half * (fl7 + fr7 + ra7);
  out[7] = half * (fl8 + fr8 + ra8);
}

// RIEMANNF / RIEMANN7F of the FP32-flux build: roe_flux's states, averages and
// waves, the dissipation in the form that FP32 resolves.
//
// |Lambda| = A1 I + D: the A1 part is A1 times the conserved jumps (R L = I);
// only D = |Lambda| - A1 I goes through the eigenvectors.  With the
// reference's form, the entropy wave and the acoustic waves carry opposite
// dp/c^2 terms that cancel, which at large Mach number (c^2 << u^2, e.g. a
// pressure on its floor) FP32 cannot resolve.  The two waves U + s and U - s of a
// kind enter as the half-sum and half-difference of their D, each formed without
// cancellation (jump_pair).
//
// The kernels around it are bound by VALU issue, so the eigenvector products
// are grouped by their shared factors, selects take the place of branches and
// a reciprocal that several quotients share is formed once.  With the limiters
// and quotients of this build (minmod32, Denom): 256^3, four fluids, the plasma's
// tile kernel 1.29 -> 1.04 ms (890 -> 650 VALU instructions per face), the neutrals'
// 1.33 -> 1.19, a step 11.9 -> 11.2 ms; 91 x 75 x 53, two fluids, van Leer, the face
// kernel 39 -> 24 us.  Errors against the FP64 flux over random states (smooth, jumps,
// Mach 20, cold, without tangential field) equal the ungrouped form's.
template <bool seven>
__device__ __forceinline__ void roe_flux32(const Consts& C, const MState<float>& L,
                                           const MState<float>& R, float* out) {
  using T = float;
  const T half = 0.5f, one = 1.f, zero = 0.f, two = 2.f;
  const T g = (T)C.gamma, hg = (T)C.hgamma;
  const T c4 = (T)k1_4PI, c8 = (T)k1_8PI, rs2 = (T)kSQRT_2;
  const Denom<T> byHg(hg, C.invhgamma), byRhoL(L.rho), byRhoR(R.rho);

  const T RUL = L.rho * L.u, RVL = L.rho * L.v, RWL = L.rho * L.w;
  const T BxBL = c8 * (L.bx * L.bx + L.by * L.by + L.bz * L.bz);
  const T RUxUL = half * (RUL * L.u + RVL * L.v + RWL * L.w);
  const T PL = L.p + BxBL;
  const T EL = byHg(L.p) + RUxUL + BxBL;
  const T AL2 = byRhoL(g * L.p);
  const T RUR = R.rho * R.u, RVR = R.rho * R.v, RWR = R.rho * R.w;
  const T BxBR = c8 * (R.bx * R.bx + R.by * R.by + R.bz * R.bz);
  const T RUxUR = half * (RUR * R.u + RVR * R.v + RWR * R.w);
  const T PR = R.p + BxBR;
  const T ER = byHg(R.p) + RUxUR + BxBR;
  const T AR2 = byRhoR(g * R.p);

  T Rho, U, V, W, BX, BY, BZ, BX2, BYZ2, BxBH, kk, cc;
  if (C.iAveraging == 1) {
    const T HL = byRhoL(EL + PL), HR = byRhoR(ER + PR);
    const T cL = __builtin_amdgcn_rcpf(one + tsqrt(byRhoL(R.rho)));
    const T cR = one - cL;
    Rho = R.rho * cL + L.rho * cR;
    U = L.u * cL + R.u * cR;
    V = L.v * cL + R.v * cR;
    W = L.w * cL + R.w * cR;
    const T HAV = HL * cL + HR * cR;
    BX = R.bx * cL + L.bx * cR;
    BY = R.by * cL + L.by * cR;
    BZ = R.bz * cL + L.bz * cR;
    const T BXAV = half * (L.bx + R.bx);
    BX2 = BXAV * BXAV;
    BYZ2 = BY * BY + BZ * BZ;
    BxBH = c8 * (BX2 + BYZ2);
    kk = half * (U * U + V * V + W * W);
    const T dbx = R.bx - L.bx, dby = R.by - L.by, dbz = R.bz - L.bz;
    const T X = byRhoL(c8 * (dbx * dbx + dby * dby + dbz * dbz) * cL * cL);
    cc = hg * (HAV - kk - Denom<T>(Rho)(c4 * (BX * BXAV + BYZ2))) + (two - g) * X;
  } else {
    Rho = half * (L.rho + R.rho);
    U = half * (L.u + R.u); V = half * (L.v + R.v); W = half * (L.w + R.w);
    BX = half * (L.bx + R.bx); BY = half * (L.by + R.by); BZ = half * (L.bz + R.bz);
    const T P = half * (PL + PR);
    BX2 = BX * BX;
    BYZ2 = BY * BY + BZ * BZ;
    BxBH = c8 * (BX2 + BYZ2);
    kk = half * (U * U + V * V + W * W);
    cc = Denom<T>(Rho)(g * (P - BxBH));
  }
  const Denom<T> byRho(Rho);
  const T bb = byRho(c4 * BX2);
  const T ccmi = tmin(AR2, AL2), ccma = tmax(AL2, AR2);
  cc = cc < ccmi ? ccmi : cc;
  cc = cc > ccma ? ccma : cc;
  const T b = tsqrt(bb), c = tsqrt(cc);

  // (BY, BZ) / |BYZ| and the fast and slow speeds
  const T sB = (T)C.smallB;
  const bool noBt = BYZ2 < sB * sB;
  const Denom<T> byHyz(tsqrt(BYZ2));
  const T hyy = noBt ? rs2 : byHyz(BY), hzz = noBt ? rs2 : byHyz(BZ);
  const T szb = cc + byRho(BxBH + BxBH);
  const T hh = tsqrt(nonneg(szb * szb - 4.f * cc * bb));
  T aas = half * (szb - hh), aaf = half * (szb + hh);
  aas = aas <= zero ? zero : (aas >= cc ? cc : aas);
  aaf = aaf <= cc ? cc : aaf;
  const bool bOver = bb > cc;
  aaf = noBt ? (bOver ? bb : cc) : aaf;
  aas = noBt ? (bOver ? cc : bb) : aas;
  const T af = tsqrt(aaf), as = tsqrt(aas);
  const T dfs = aaf - aas, cs = cc - aas, fc = aaf - cc;
  const Denom<T> byDfs(dfs);
  T alf = tsqrt(byDfs(cs)), als = tsqrt(byDfs(fc));
  const bool fast = dfs < 1.0e-8f, slow = !fast && cs <= zero, fast2 = fast || fc <= zero;
  alf = slow ? zero : (fast2 ? one : alf);
  als = slow ? one : (fast2 ? zero : als);
  const T sih = BX >= zero ? one : -one;

  // |lambda| with the entropy fix: A1 = |U| fixed, and per kind of wave of speed
  // s the sum and the difference of D(U + s) and D(U - s)
  const T del = (T)C.del2 * (fabs(U) + fabs(V) + fabs(W) + af);
  const T hdel = half * del, hid = half * __builtin_amdgcn_rcpf(del);
  const T aU = fabs(U), sU = U >= zero ? one : -one;
  const bool ge = aU >= del;
  const T A1 = ge ? aU : aU * aU * hid + hdel;
  auto jump_pair = [&](T s, T& sum, T& dif) {
    const T tp = aU + s, tm = aU - s, zm = fabs(tm);
    const T up = ge ? s : (tp >= del ? tp - A1 : s * (aU + tp) * hid);
    const T fm = zm >= del ? zm - A1 : zm * zm * hid + hdel - A1;
    const T dn = ge ? (tm >= del ? -s : fm) : (zm < del ? -s * (aU + tm) * hid : fm);
    sum = up + dn;
    dif = sU * (up - dn);
  };
  T sa, da, sf, df, ss, ds;
  jump_pair(b, sa, da);
  jump_pair(af, sf, df);
  jump_pair(as, ss, ds);

  T du[8], dcons[8];
  roe_jumps<T, seven>(C, L, R, byRho, U, V, W, BX, BY, BZ, kk, du, dcons);
  const T sq = tsqrt((T)kPI * Rho), sq2 = two * rs2 * sq;
  const T isq = __builtin_amdgcn_rcpf(sq), ic = __builtin_amdgcn_rcpf(cc);
  const T hic = half * ic, aff = alf * af, ass = als * as;
  // left eigenvectors times the jumps
  const T Pa = rs2 * (hyy * du[3] - hzz * du[2]);
  const T Qa = half * rs2 * isq * sih * (hzz * du[6] - hyy * du[7]);
  const T vt = sih * (hyy * du[2] + hzz * du[3]);
  const T Xf = hic * (aff * du[1] - ass * vt), Xs = hic * (ass * du[1] + aff * vt);
  const T P5 = byRho(hic * du[4]), Bt = 0.25f * ic * c * isq * (hyy * du[6] + hzz * du[7]);
  const T Yf = alf * P5 + als * Bt, Ys = als * P5 - alf * Bt;
  // D of the waves, and the right eigenvectors
  const T lp = rs2 * (sa * Pa + da * Qa), lm = sih * sq2 * (sa * Qa + da * Pa);
  const T s56 = df * Xf + sf * Yf, m56 = sf * Xf + df * Yf;
  const T s78 = ds * Xs + ss * Ys, m78 = ss * Xs + ds * Ys;
  const T M = sih * (aff * m78 - ass * m56);
  const T N = two * sq * c * (als * s56 - alf * s78);
  T ra1 = Rho * (alf * s56 + als * s78);
  T ra2 = aff * m56 + ass * m78;
  T ra3 = hyy * M - hzz * lp;
  T ra4 = hzz * M + hyy * lp;
  T ra7 = hzz * lm + hyy * N;
  T ra8 = hzz * N - hyy * lm;
  T ra5 = ra1 * kk + Rho * (U * ra2 + V * ra3 + W * ra4) + byHg(cc * ra1) +
          c4 * (BY * ra7 + BZ * ra8);
  ra2 = U * ra1 + Rho * ra2 + A1 * dcons[1];
  ra3 = V * ra1 + Rho * ra3 + A1 * dcons[2];
  ra4 = W * ra1 + Rho * ra4 + A1 * dcons[3];
  ra1 = ra1 + A1 * dcons[0];
  ra5 = ra5 + A1 * dcons[4];
  ra7 = ra7 + A1 * dcons[6];
  ra8 = ra8 + A1 * dcons[7];

  const T fl2 = L.u * RUL - L.bx * L.bx * c4 + PL;
  const T fr2 = R.u * RUR - R.bx * R.bx * c4 + PR;
  const T fl3 = L.u * RVL - L.bx * L.by * c4, fr3 = R.u * RVR - R.bx * R.by * c4;
  const T fl4 = L.u * RWL - L.bx * L.bz * c4, fr4 = R.u * RWR - R.bx * R.bz * c4;
  const T fl5 = L.u * (EL + PL) - L.bx * (L.u * L.bx + L.v * L.by + L.w * L.bz) * c4;
  const T fr5 = R.u * (ER + PR) - R.bx * (R.u * R.bx + R.v * R.by + R.w * R.bz) * c4;
  const T fl7 = L.u * L.by - L.bx * L.v, fr7 = R.u * R.by - R.bx * R.v;
  const T fl8 = L.u * L.bz - L.bx * L.w, fr8 = R.u * R.bz - R.bx * R.w;
  out[0] = half * (RUL + RUR + ra1);
  out[1] = half * (fl2 + fr2 + ra2);
  out[2] = half * (fl3 + fr3 + ra3);
  out[3] = half * (fl4 + fr4 + ra4);
  out[4] = half * (fl5 + fr5 + ra5);
  out[5] = seven ? zero : half * (A1 * dcons[5]);
  out[6] = half * (fl7 + fr7 + ra7);
  out[7] = half * (fl8 + fr8 + ra8);
}

// Rusanov flux (RUSANOVF, src/RusanovF.ChF:4-197)
template <typename T>
__device__ __forceinline__ void rusanov_flux(const Consts& C,
                                             const MState<T>& L,
                                             const MState<T>& R, T* out) {
  const T half = T(0.5), one = T(1), two = T(2);
  const T g = T(C.gamma), hg = T(C.hgamma);
  const T c4 = T(k1_4PI), c8 = T(k1_8PI);
  const Denom<T> byHg(hg, C.invhgamma);
  const T RUL = L.rho * L.u, RVL = L.rho * L.v, RWL = L.rho * L.w;
  const T BxBL = c8 * (L.bx * L.bx + L.by * L.by + L.bz * L.bz);
  const T RUxUL = half * (RUL * L.u + RVL * L.v + RWL * L.w);
  const T PL = L.p + BxBL, EL = byHg(L.p) + RUxUL + BxBL;
  const T BXL4 = L.bx * c4;
  const T RUR = R.rho * R.u, RVR = R.rho * R.v, RWR = R.rho * R.w;
  const T BxBR = c8 * (R.bx * R.bx + R.by * R.by + R.bz * R.bz);
  const T RUxUR = half * (RUR * R.u + RVR * R.v + RWR * R.w);
  const T PR = R.p + BxBR, ER = byHg(R.p) + RUxUR + BxBR;
  const T BXR4 = R.bx * c4;
  T Rho, U, BX2, BxBH, A2;
  if (C.iAveraging == 1) {
    const Denom<T> byRhoL(L.rho), byRhoR(R.rho);
    const T HL = byRhoL(EL + PL), HR = byRhoR(ER + PR);
    const T cL = Denom<T>(one + tsqrt(byRhoL(R.rho)))(one);
    const T cR = one - cL;
    Rho = R.rho * cL + L.rho * cR;
    U = L.u * cL + R.u * cR;
    const T V = L.v * cL + R.v * cR, W = L.w * cL + R.w * cR;
    const T HAV = HL * cL + HR * cR;
    const T BX = R.bx * cL + L.bx * cR, BY = R.by * cL + L.by * cR,
            BZ = R.bz * cL + L.bz * cR;
    const T BXAV = half * (L.bx + R.bx);
    BX2 = BXAV * BXAV;
    const T BYZ2 = BY * BY + BZ * BZ;
    BxBH = c8 * (BX2 + BYZ2);
    const T kk = half * (U * U + V * V + W * W);
    const T dbx = R.bx - L.bx, dby = R.by - L.by, dbz = R.bz - L.bz;
    const T X = byRhoL(c8 * (dbx * dbx + dby * dby + dbz * dbz) * cL * cL);
    A2 = hg * (HAV - kk - Denom<T>(Rho)(c4 * (BX * BXAV + BYZ2))) + (two - g) * X;
  } else {
    Rho = half * (L.rho + R.rho);
    U = half * (L.u + R.u);
    const T BX = half * (L.bx + R.bx), BY = half * (L.by + R.by),
            BZ = half * (L.bz + R.bz);
    const T PGas = half * (L.p + R.p);
    BX2 = BX * BX;
    BxBH = c8 * (BX2 + BY * BY + BZ * BZ);
    A2 = Denom<T>(Rho)(g * PGas);
  }
  const Denom<T> byRho(Rho);
  const T bb = byRho(c4 * BX2);
  const T szb = A2 + byRho(BxBH + BxBH);
  const T hh = tsqrt(nonneg(szb * szb - T(4) * A2 * bb));
  const T af = tsqrt(half * (szb + hh));
  const T em = fabs(U) + af;
  out[0] = half * (RUL + RUR + em * (L.rho - R.rho));
  out[1] = half * ((L.u * RUL - BXL4 * L.bx + PL) + (R.u * RUR - BXR4 * R.bx + PR) +
                   em * (RUL - RUR));
  out[2] = half * ((L.u * RVL - BXL4 * L.by) + (R.u * RVR - BXR4 * R.by) +
                   em * (RVL - RVR));
  out[3] = half * ((L.u * RWL - BXL4 * L.bz) + (R.u * RWR - BXR4 * R.bz) +
                   em * (RWL - RWR));
  out[4] = half * ((L.u * (EL + PL) - BXL4 * (L.u * L.bx + L.v * L.by + L.w * L.bz)) +
                   (R.u * (ER + PR) - BXR4 * (R.u * R.bx + R.v * R.by + R.w * R.bz)) +
                   em * (EL - ER));
  out[5] = half * (T(0) + T(0) + em * (L.bx - R.bx));
  out[6] = half * ((L.u * L.by - L.bx * L.v) + (R.u * R.by - R.bx * R.v) +
                   em * (L.by - R.by));
  out[7] = half * ((L.u * L.bz - L.bx * L.w) + (R.u * R.bz - R.bx * R.w) +
                   em * (L.bz - R.bz));
}

// HLLC flux of ideal MHD (S. Li, J. Comput. Phys. 203 (2005) 344-357), in
// the reference's Gaussian units (magnetic pressure B^2/8pi, Maxwell
// stress B B/4pi).  No counterpart in the reference's solvers.  Outer
// speeds S_L = min(u_L - c_fL, u_R - c_fR), S_R = max(u_L + c_fL,
// u_R + c_fR) (normal fast speeds); the star region takes the HLL state's
// field B* = B_hll and contact speed S_M = (rho u)_hll / rho_hll, the total
// pressure p_T* = rho_L (S_L - u_L)(S_M - u_L) + p_TL - (B_xL^2 - B_x*^2)/4pi,
// and on each side K
//   rho*_K = rho_K (S_K - u_K) / (S_K - S_M),   (rho u)*_K = rho*_K S_M,
//   (rho v_t)*_K = [rho_K v_tK (S_K - u_K) - (B_x* B_t* - B_xK B_tK)/4pi] / (S_K - S_M),
//   E*_K = [E_K (S_K - u_K) - p_TK u_K + p_T* S_M
//           + (B_xK (v_K . B_K) - B_x* (v* . B*))/4pi] / (S_K - S_M),
// v* = (S_M, v_hll, w_hll); F = F_K + S_K (U*_K - U_K) on the side of the
// contact that holds x/t = 0, F_L or F_R beyond the outer waves.  Inputs
// clamped to (smallp, smallr) like the other solvers'; out order as
// roe_flux's.
template <typename T>
__device__ __forceinline__ void hllc_flux(const Consts& C, const MState<T>& L,
                                          const MState<T>& R, T* out) {
  const T half = T(0.5), zero = T(0);
  const T g = T(C.gamma), hg = T(C.hgamma);
  const T c4 = T(k1_4PI), c8 = T(k1_8PI);
  const Denom<T> byHg(hg, C.invhgamma);
  // conserved states and physical fluxes of both sides
  T UL[8], UR[8], FL[8], FR[8];
  T ptL, ptR;
  {
    const T b2 = L.bx * L.bx + L.by * L.by + L.bz * L.bz;
    ptL = L.p + c8 * b2;
    const T E = byHg(L.p) + half * L.rho * (L.u * L.u + L.v * L.v + L.w * L.w) + c8 * b2;
    const T vb = L.u * L.bx + L.v * L.by + L.w * L.bz;
    UL[0] = L.rho; UL[1] = L.rho * L.u; UL[2] = L.rho * L.v; UL[3] = L.rho * L.w;
    UL[4] = E; UL[5] = L.bx; UL[6] = L.by; UL[7] = L.bz;
    FL[0] = UL[1];
    FL[1] = UL[1] * L.u + ptL - c4 * L.bx * L.bx;
    FL[2] = UL[1] * L.v - c4 * L.bx * L.by;
    FL[3] = UL[1] * L.w - c4 * L.bx * L.bz;
    FL[4] = (E + ptL) * L.u - c4 * L.bx * vb;
    FL[5] = zero;
    FL[6] = L.u * L.by - L.v * L.bx;
    FL[7] = L.u * L.bz - L.w * L.bx;
  }
  {
    const T b2 = R.bx * R.bx + R.by * R.by + R.bz * R.bz;
    ptR = R.p + c8 * b2;
    const T E = byHg(R.p) + half * R.rho * (R.u * R.u + R.v * R.v + R.w * R.w) + c8 * b2;
    const T vb = R.u * R.bx + R.v * R.by + R.w * R.bz;
    UR[0] = R.rho; UR[1] = R.rho * R.u; UR[2] = R.rho * R.v; UR[3] = R.rho * R.w;
    UR[4] = E; UR[5] = R.bx; UR[6] = R.by; UR[7] = R.bz;
    FR[0] = UR[1];
    FR[1] = UR[1] * R.u + ptR - c4 * R.bx * R.bx;
    FR[2] = UR[1] * R.v - c4 * R.bx * R.by;
    FR[3] = UR[1] * R.w - c4 * R.bx * R.bz;
    FR[4] = (E + ptR) * R.u - c4 * R.bx * vb;
    FR[5] = zero;
    FR[6] = R.u * R.by - R.v * R.bx;
    FR[7] = R.u * R.bz - R.w * R.bx;
  }
  // normal fast speeds: c_f^2 = (a^2 + b^2 + sqrt((a^2 + b^2)^2 - 4 a^2 b_n^2)) / 2
  auto cfast = [&](const MState<T>& S) {
    const Denom<T> byRho(S.rho);
    const T a2 = byRho(g * S.p);
    const T b2 = byRho(c4 * (S.bx * S.bx + S.by * S.by + S.bz * S.bz));
    const T bn2 = byRho(c4 * S.bx * S.bx);
    const T s = a2 + b2;
    return tsqrt(half * (s + tsqrt(tmax(zero, s * s - T(4) * a2 * bn2))));
  };
  const T cfL = cfast(L), cfR = cfast(R);
  const T SL = tmin(L.u - cfL, R.u - cfR), SR = tmax(L.u + cfL, R.u + cfR);
  if (SL >= zero) {
#pragma unroll
    for (int c = 0; c < 8; ++c) out[c] = FL[c];
    return;
  }
  if (SR <= zero) {
#pragma unroll
    for (int c = 0; c < 8; ++c) out[c] = FR[c];
    return;
  }
  // the HLL state (rounded as divisions: the FP64 build gives the oracle's
  // bits)
  const Denom<T> bySpan(SR - SL);
  T H[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) H[c] = bySpan(SR * UR[c] - SL * UL[c] - (FR[c] - FL[c]));
  const Denom<T> byH0(H[0]);
  const T SM = byH0(H[1]);
  const T vh = byH0(H[2]), wh = byH0(H[3]);
  const T bx = H[5], hy = H[6], bz = H[7];
  const T ptS = L.rho * (SL - L.u) * (SM - L.u) + ptL - c4 * (L.bx * L.bx - bx * bx);
  const bool left = SM >= zero;
  const MState<T>& K = left ? L : R;
  const T* UK = left ? UL : UR;
  const T* FK = left ? FL : FR;
  const T SK = left ? SL : SR, ptK = left ? ptL : ptR;
  const T sk = SK - K.u;
  // left of the contact both sides of the quotients are negative: over a
  // positive denominator a zero numerator gives the division's sign
  const T sg = left ? T(-1) : T(1);
  const Denom<T> by(sg * (SK - SM));
  T S[8];
  S[0] = by(sg * (K.rho * sk));
  S[1] = S[0] * SM;
  S[2] = by(sg * (K.rho * K.v * sk - c4 * (bx * hy - K.bx * K.by)));
  S[3] = by(sg * (K.rho * K.w * sk - c4 * (bx * bz - K.bx * K.bz)));
  S[4] = by(sg * (UK[4] * sk - ptK * K.u + ptS * SM +
                  c4 * (K.bx * (K.u * K.bx + K.v * K.by + K.w * K.bz) -
                        bx * (SM * bx + vh * hy + wh * bz))));
  S[5] = bx; S[6] = hy; S[7] = bz;
#pragma unroll
  for (int c = 0; c < 8; ++c) out[c] = FK[c] + SK * (S[c] - UK[c]);
}

// van Leer flux-vector splitting for one neutral fluid (VANLEERF /
// VANLEERRS, src/VanLeerRSF.ChF:4-240).  Inputs rotated, already clamped:
// p, rho, un, ut1, ut2.  out: rho, mn, mt1, mt2, E.
template <typename T>
__device__ __forceinline__ void vanleer_flux(const Consts& C, T pL, T rL, T uL,
                                             T vL, T wL, T pR, T rR, T uR,
                                             T vR, T wR, T* out) {
  const T g = T(C.gamma), hg = T(C.hgamma), half = T(0.5), zero = T(0);
  const Denom<T> byHg(hg, C.invhgamma), byG(g, C.invgamma);
  T p1, p2, p3, p4, p5;  // F+ from the left state
  {
    const T RUxU = half * (rL * uL * uL + rL * vL * vL + rL * wL * wL);
    const T E = byHg(pL) + RUxU;
    const Denom<T> byRho(rL);
    const T a = tsqrt(byRho(g * pL));
    if (uL <= -a) { p1 = p2 = p3 = p4 = p5 = zero; }
    else if (uL >= a) {
      p1 = rL * uL; p2 = p1 * uL + pL; p3 = p1 * vL; p4 = p1 * wL;
      p5 = uL * (E + pL);
    } else {
      const T UA = byG(-uL + (a + a));
      const T H = byRho(E + pL);
      const T HU = uL + a;
      p1 = Denom<T>(a)(T(0.25) * rL * HU * HU);
      p2 = p1 * (uL + UA); p3 = p1 * vL; p4 = p1 * wL; p5 = p1 * H;
    }
  }
  T m1, m2, m3, m4, m5;  // F- from the right state
  {
    const T RUxU = half * (rR * uR * uR + rR * vR * vR + rR * wR * wR);
    const T E = byHg(pR) + RUxU;
    const Denom<T> byRho(rR);
    const T a = tsqrt(byRho(g * pR));
    if (uR >= a) { m1 = m2 = m3 = m4 = m5 = zero; }
    else if (uR <= -a) {
      m1 = rR * uR; m2 = m1 * uR + pR; m3 = m1 * vR; m4 = m1 * wR;
      m5 = uR * (E + pR);
    } else {
      const T UA = byG(-uR - (a + a));
      const T H = byRho(E + pR);
      const T HU = uR - a;
      m1 = Denom<T>(a)(-T(0.25) * rR * HU * HU);
      m2 = m1 * (uR + UA); m3 = m1 * vR; m4 = m1 * wR; m5 = m1 * H;
    }
  }
  out[0] = m1 + p1; out[1] = m2 + p2; out[2] = m3 + p3; out[3] = m4 + p4;
  out[4] = m5 + p5;
}

}  // namespace mfm
