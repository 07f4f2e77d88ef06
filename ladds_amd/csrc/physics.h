// physics.h -- device force model of the Yoshida propagator.
//
// Replaces OrbitPropagator's AccelerationAccumulator and its eight components
// (upstream FG-TUM/OrbitPropagator @ b90f3bae, selected by the flag array built at
// src/ladds/Simulation.cpp:127-135).  The upstream source is not part of the
// LADDS tree, so each component is restated from its published form:
//   KEP, J2, C22, S22  Montenbruck & Gill, Satellite Orbits (2000) Sec. 3.2
//   SOL, LUN           third-body term, M&G eq. 3.37
//   SRP                cannonball model, M&G eq. 3.75, cylindrical shadow (Sec. 3.4.2)
//   DRAG               M&G eq. 3.97 with a co-rotating atmosphere and the exponential
//                      density table of Vallado (2013) Table 8-4
// evasivePreserving objects receive the Keplerian term only (Particle.h:49-52).
//
// Precision forms:
//   kFormFp64      every term in FP64.  Third-body and SRP use the direct form
//                  GM (d/|d|^3 - s/|s|^3): its cancellation costs ~1e-12 relative in FP64.
//   kFormSplit     Kepler, J2, C22/S22 and drag in FP64; Sun, Moon and SRP in FP32,
//                  accumulated into the FP64 kick.  J2's acceleration needs ~29
//                  significant bits to hold 1 cm/day (FP32 has 24), and drag moves a
//                  low object hundreds of km along-track per day, so FP32 rounding of
//                  either costs centimetres (measured: up to 1 m for J2, 25 cm for drag).
//                  The tesseral terms in FP32 (Earth-fixed rotation and field) leave
//                  0.5 cm at the 99.9th percentile and over 1 cm in the tail of a
//                  1M-object day, so they stay FP64 too; the FP32 terms then contribute
//                  ~0.01 cm.  The FP32 third-body terms use Battin's cancellation-free
//                  form a = -GM/|s|^3 (1+q)^-3/2 (r + f(q) s) (Battin 1987, eq. 8.61).
//                  The SRP shadow decision is taken on the FP64 state.
//   kFormSplitAll32  J2, C22/S22, Sun, Moon and SRP in FP32 (Kepler and drag FP64).
#pragma once

#include <hip/hip_runtime.h>

#include "constants.h"
#include "engine.h"

namespace ladds {

enum : unsigned {
  kKepBit = 1u << 0,
  kJ2Bit = 1u << 1,
  kC22Bit = 1u << 2,
  kS22Bit = 1u << 3,
  kSolBit = 1u << 4,
  kLunBit = 1u << 5,
  kSrpBit = 1u << 6,
  kDragBit = 1u << 7,
  kAllBits = 0xFFu
};

// Exponential atmosphere staged in LDS by the kernels.  Every row begins at a multiple of
// 5 km, so the row of an altitude is one table read at its 5 km bin (a binary search over
// the 28 rows was five dependent LDS reads and ~15 more instructions per evaluation).
constexpr int kAtmBins = 201;  // 5 km bins from 0 to 1000 km (the last one: above 1000 km)
constexpr double kAtmBinKm = 5.0;
struct alignas(16) AtmRow {
  double h0, inv_scale, rho, pad;
};
struct AtmTable {
  AtmRow row[kAtmRows];
  uint8_t bin[(kAtmBins + 7) / 8 * 8];
};
static_assert(sizeof(AtmTable) % sizeof(double) == 0, "staged as doubles");

// Host-side fill of the table from the constants (uploaded to __constant__ memory by the
// kernels' translation units).
inline void fill_atm_table(AtmTable &t) {
  for (int i = 0; i < kAtmRows; ++i) t.row[i] = AtmRow{kAtmH0[i], 1.0 / kAtmScale[i], kAtmRho[i], 0.0};
  for (int b = 0; b < (int)sizeof(t.bin); ++b) {
    int i = 0;
    while (i + 1 < kAtmRows && kAtmH0[i + 1] <= kAtmBinKm * b) ++i;
    t.bin[b] = (uint8_t)i;
  }
}

// 1/sqrt(x) of a positive x from the hardware's estimate y (~2^-24), one step of third order
// (Householder's iteration): y (1 + e/2 + 3 e^2/8) with e = 1 - x y^2, which leaves rounding
// error only.
__device__ __forceinline__ double rsqrt64_step(double x, double y) {
  const double e = fma(-x * y, y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
}

// FAR: x may have overflowed and then gives 0 (its estimate; e is formed with a finite x).  Paid
// by every object that took 2% of 1,000 steps of 250,007, so the propagation's paths for the
// usual models go without and leave the objects beyond kFar to the general one.  (On the high
// word alone: a 64-bit constant would take scalar registers, which spill there and cost the
// other paths of the split form 11 instructions a step.)
template <bool FAR>
__device__ __forceinline__ double rsqrt64(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  if (FAR) x = __hiloint2double((int)min((unsigned)__double2hiint(x), 0x7FEFFFFFu), __double2loint(x));
  return rsqrt64_step(x, y);
}

// An object whose coordinates [km] sum up to less at the start of a launch does not come near the
// overflow of its squared distances within it.
constexpr double kFar = 0x1p465;  // ~1e140

// a b + c with c a constant of the loop.  Written out because the compiler picks the two-address
// form here and copies the constant into its destination first, one more instruction each.
__device__ __forceinline__ double fma_const(double a, double b, double c) {
  double d;
  asm("v_fma_f64 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "v"(c));
  return d;
}

// exp(x), x < 1000 (below -1500, and for NaN, exp(-1500) = 0): x = n ln 2 + r, and
// exp(r) = 1 + r + r^2 q(r) with q the degree-9 Chebyshev interpolant on |r| <= ln(2)/2
// (relative error 2e-17), its even and odd halves evaluated side by side.
__device__ __forceinline__ double exp64(double x) {
  const double u = fmax(x, -1500.0);
  const double n = rint(u * 1.4426950408889634);
  const double r = fma(n, -2.3190468138462996e-17, fma(n, -0.6931471805599453, u));
  const double r2 = r * r;
  double even = fma_const(2.7620075879983367e-07, r2, 2.4801521322368692e-05);
  double odd = fma_const(2.5100375832561234e-08, r2, 2.7557268480310024e-06);
  even = fma_const(even, r2, 0.0013888888917196719);
  odd = fma_const(odd, r2, 0.00019841269863040545);
  even = fma_const(even, r2, 0.041666666666624164);
  odd = fma_const(odd, r2, 0.008333333333330065);
  even = fma_const(even, r2, 0.5000000000000001);
  odd = fma_const(odd, r2, 0.16666666666666669);
  return __builtin_ldexp(fma(r2, fma(odd, r, even), r) + 1.0, (int)n);
}

// Row of the table: largest i with h0[i] <= h (0 below the table).  h / 5 km can round up to
// the next bin just below its edge; the remainder's sign shows it.  h is above -R_E, and
// altitudes above the table (and NaN) read its last bin.
__device__ __forceinline__ const AtmRow &atm_row(double h, const AtmTable &t) {
  const double hc = fmin(h, kAtmBinKm * (kAtmBins - 1));
  const double b = floor(hc * (1.0 / kAtmBinKm));
  int i = (int)b;
  if (fma(-kAtmBinKm, b, hc) < 0.0) i -= 1;
  return t.row[t.bin[max(i, 0)]];
}

// rho0[i] * exp(-(h - h0[i]) / H[i]) in FP64.
__device__ __forceinline__ double atm_density(double h, const AtmTable &t) {
  const AtmRow &row = atm_row(h, t);
  return row.rho * exp64((row.h0 - h) * row.inv_scale);
}

// Tesseral degree-2 order-2 terms.  In the Earth-fixed frame U = (kC (x^2 - y^2) + kS x y) / r^5;
// turned back by the rotation angle th it keeps that form, U = (a (x^2 - y^2) + b x y) / r^5 with
//   a = kC cos 2th - kS/2 sin 2th,  b = 2 kC sin 2th + kS cos 2th,
// so no position or acceleration is rotated.
template <typename T>
__device__ __forceinline__ void tesseral_coefficients(const SubstepEnv<T> &e, unsigned mask, T &a, T &b) {
#pragma clang fp contract(on)
  const T kc = (mask & kC22Bit) ? (T)kC22Coef : (T)0;
  const T ks = (mask & kS22Bit) ? (T)kS22Coef : (T)0;
  a = kc * e.c2 - (T)0.5 * ks * e.s2;
  b = (T)2 * kc * e.s2 + ks * e.c2;
}

// Adds the gradient of U.
template <typename T>
__device__ __forceinline__ void tesseral(T x, T y, T z, T inv_r2, T inv_r5, T a, T b, T &ax, T &ay, T &az) {
#pragma clang fp contract(on)
  const T u = a * ((x - y) * (x + y)) + b * (x * y);
  const T q = (T)-5 * u * (inv_r5 * inv_r2);
  const T gx = ((T)2 * a * x + b * y) * inv_r5 + q * x;
  const T gy = (b * x - (T)2 * a * y) * inv_r5 + q * y;
  const T gz = q * z;
  ax += gx;
  ay += gy;
  az += gz;
}

// Cylindrical shadow test (M&G Sec. 3.4.2), always in FP64: it is a discontinuous
// decision, so it is taken on the FP64 state in every precision form.
__device__ __forceinline__ bool in_shadow(double x, double y, double z, double r2, const SubstepEnv<double> &e) {
#pragma clang fp contract(on)
  const double rs = x * e.sun[0] + y * e.sun[1] + z * e.sun[2];
  return (rs < 0.0) && (r2 - rs * rs * e.sun_inv_s2 < kREarth * kREarth);
}

// Environments of one step, copied to LDS by the wavefront that reads them: lane l moves word
// l.  Few wavefronts per SIMD cannot hide the scalar loads of environments that no other
// wavefront of their XCD has read yet; fetched a step ahead they cost nothing.
struct EnvStage {
  SubstepEnv<double> e64[3];
  SubstepEnv<float> e32[3];
};
constexpr int kEnvWords64 = 3 * (int)sizeof(SubstepEnv<double>) / 8;  // 60
constexpr int kEnvWords32 = 3 * (int)sizeof(SubstepEnv<float>) / 8;   // 30
static_assert(kEnvWords64 <= 64 && kEnvWords32 <= 64, "one word per lane");

// FP64 third body, direct form GM d/|d|^3 - GM s/|s|^3 with d = s - r; returns 1/|d|^3.
template <bool FAR>
__device__ __forceinline__ double third_body64(double dx, double dy, double dz, double gm, const double *acc,
                                               bool gravity, double &ax, double &ay, double &az) {
#pragma clang fp contract(off)
  const double inv_d = rsqrt64<FAR>(fma(dz, dz, fma(dx, dx, dy * dy)));
  const double inv_d3 = inv_d * inv_d * inv_d;
  if (gravity) {
    const double f = gm * inv_d3;
    ax += fma(f, dx, -acc[0]);
    ay += fma(f, dy, -acc[1]);
    az += fma(f, dz, -acc[2]);
  }
  return inv_d3;
}

// FP32 third body (Battin's form) and, sharing its geometry, SRP for the Sun.
// k = GM/|s|^3; inv_p32 = (1+q)^{-3/2} = |s|^3 / |r - s|^3.
template <bool SUN>
__device__ __forceinline__ void third_body32(float x, float y, float z, float r2, const float *s, float inv_s2,
                                             float k, bool gravity, bool radiation, float srp, float &ax, float &ay,
                                             float &az) {
#pragma clang fp contract(off)
  const float rs = fmaf(z, s[2], fmaf(x, s[0], y * s[1]));
  const float t = fmaf(-2.f, rs, r2);
  const float q = t * inv_s2;
  const float onepq = fmaf(t, inv_s2, 1.f);
  const float rq = __builtin_amdgcn_rsqf(onepq);
  const float inv_p32 = rq * rq * rq;
  if (gravity) {
    const float p1 = fmaf(onepq * onepq, rq, 1.f);  // 1 + (1+q)^{3/2}
    const float q3 = SUN ? q + 3.f : fmaf(t, inv_s2, 3.f);
    const float f = q * fmaf(q, q3, 3.f) * __builtin_amdgcn_rcpf(p1);
    const float kk = k * inv_p32;
    ax = fmaf(-kk, fmaf(f, s[0], x), ax);
    ay = fmaf(-kk, fmaf(f, s[1], y), ay);
    az = fmaf(-kk, fmaf(f, s[2], z), az);
  }
  if (SUN && radiation) {
    // 1/|r - s|^3 = (k / GM_sun) (1+q)^{-3/2}
    const float g = srp * (k * (float)(1.0 / kGmSun)) * inv_p32;
    ax = fmaf(g, x - s[0], ax);
    ay = fmaf(g, y - s[1], ay);
    az = fmaf(g, z - s[2], az);
  }
}

// Drag with a co-rotating atmosphere; drag64 = kDragCoef * bc_inv.
__device__ __forceinline__ void drag_term64(double x, double y, double vx, double vy, double vz, double h,
                                            double drag64, const AtmTable &t, double &ax, double &ay, double &az) {
#pragma clang fp contract(off)
  const double om = kOmegaEarth;
  const double wx = fma(om, y, vx), wy = fma(-om, x, vy), wz = vz;
  const double w2 = fma(wz, wz, fma(wx, wx, wy * wy));
  const double vn = w2 * rsqrt64<false>(fmax(w2, 1e-290));  // 0 without wind
  const double f = drag64 * atm_density(h, t) * vn;
  ax = fma(f, wx, ax);
  ay = fma(f, wy, ay);
  az = fma(f, wz, az);
}

struct ObjParams {
  double srp64, drag64;
  float srp32;
  int activity;
};

// Acceleration [km/s^2] of one object in the given precision form.  Called with a constant
// mask where that holds for the whole wavefront, so that the components' dependent chains
// interleave; else `mask` may differ from lane to lane (evasivePreserving objects).
//
// Products and sums are fused where the code says so and nowhere else: every instantiation
// rounds alike, and the components are added one after the other, Kepler first.  Merged into
// one factor on the position they would cost ~10 instructions fewer, but a differently rounded
// Kepler or J2 term shows in a pair's squared distance after some hundred steps (3e-9
// relative after four hours).  SRP shares the Sun's geometry.  FAR: see rsqrt64.
template <int FORM, bool FAR>
__device__ __forceinline__ void acceleration(double x, double y, double z, double vx, double vy, double vz,
                                             const ObjParams &p, unsigned mask, const SubstepEnv<double> &e64,
                                             const SubstepEnv<float> &e32, const AtmTable &atm, double &ax,
                                             double &ay, double &az) {
#pragma clang fp contract(off)
  const double r2 = fma(z, z, fma(x, x, y * y));
  const double inv_r = rsqrt64<FAR>(r2);
  const double inv_r2 = inv_r * inv_r;
  const double inv_r3 = inv_r2 * inv_r;
  // (chosen, not multiplied by 0: without this force an object at the origin, or infinitely far, has none)
  const bool kepler = (mask & kKepBit) != 0u;
  const double fk = -kMuEarth * inv_r3;
  ax = kepler ? fk * x : 0.0;
  ay = kepler ? fk * y : 0.0;
  az = kepler ? fk * z : 0.0;
  constexpr bool j2_64 = (FORM != kFormSplitAll32);
  constexpr bool tess_64 = (FORM != kFormSplitAll32);
  const double inv_r5 = inv_r3 * inv_r2;
  if (j2_64 && (mask & kJ2Bit)) {
    const double t = z * z * inv_r2;  // z2 = 5 t
    const double f = -kJ2Coef * inv_r3 * inv_r2;
    const double one = fma(-5.0, t, 1.0);
    ax = fma(f * x, one, ax);
    ay = fma(f * y, one, ay);
    az = fma(f * z, fma(-5.0, t, 3.0), az);
  }
  // drag in FP64 in every form
  if (mask & kDragBit) drag_term64(x, y, vx, vy, vz, fma(r2, inv_r, -kREarth), p.drag64, atm, ax, ay, az);
  if (tess_64 && (mask & (kC22Bit | kS22Bit))) {
    double a, b;
    tesseral_coefficients(e64, mask, a, b);
    tesseral(x, y, z, inv_r2, inv_r5, a, b, ax, ay, az);
  }
  if constexpr (FORM == kFormFp64) {
    double dx = 0.0, dy = 0.0, dz = 0.0, srp = 0.0;
    if (mask & (kSolBit | kSrpBit)) {
      dx = e64.sun[0] - x;
      dy = e64.sun[1] - y;
      dz = e64.sun[2] - z;
      const double inv_d3 = third_body64<FAR>(dx, dy, dz, kGmSun, e64.sun_acc, (mask & kSolBit) != 0, ax, ay, az);
      if (mask & kSrpBit) srp = (in_shadow(x, y, z, r2, e64) ? 0.0 : -p.srp64) * inv_d3;
    }
    if (mask & kLunBit)
      third_body64<FAR>(e64.moon[0] - x, e64.moon[1] - y, e64.moon[2] - z, kGmMoon, e64.moon_acc, true, ax, ay, az);
    if (mask & kSrpBit) {  // srp (r - s)/|r - s|^3
      ax = fma(srp, dx, ax);
      ay = fma(srp, dy, ay);
      az = fma(srp, dz, az);
    }
  } else {
    constexpr unsigned kFp64Bits = kKepBit | kDragBit | (j2_64 ? kJ2Bit : 0u) | (tess_64 ? (kC22Bit | kS22Bit) : 0u);
    if (mask & ~kFp64Bits) {
      const float xf = (float)x, yf = (float)y, zf = (float)z;
      const float r2f = (float)r2;
      float fx = 0.f, fy = 0.f, fz = 0.f;
      if constexpr (!j2_64) {
        const float inv_r2f = (float)inv_r2;
        const float inv_r5f = (float)inv_r3 * inv_r2f;
        if (mask & kJ2Bit) {
          const float t = zf * zf * inv_r2f;
          const float f = -(float)kJ2Coef * inv_r5f;
          const float one = fmaf(-5.f, t, 1.f);
          fx = f * xf * one;
          fy = f * yf * one;
          fz = f * zf * fmaf(-5.f, t, 3.f);
        }
        if (mask & (kC22Bit | kS22Bit)) {
          float a, b;
          tesseral_coefficients(e32, mask, a, b);
          tesseral(xf, yf, zf, inv_r2f, inv_r5f, a, b, fx, fy, fz);
        }
      }
      if (mask & (kSolBit | kSrpBit)) {
        const float srp = ((mask & kSrpBit) && !in_shadow(x, y, z, r2, e64)) ? p.srp32 : 0.f;
        third_body32<true>(xf, yf, zf, r2f, e32.sun, e32.sun_inv_s2, e32.sun_k, (mask & kSolBit) != 0,
                           (mask & kSrpBit) != 0, srp, fx, fy, fz);
      }
      if (mask & kLunBit)
        third_body32<false>(xf, yf, zf, r2f, e32.moon, e32.moon_inv_s2, e32.moon_k, true, false, 0.f, fx, fy, fz);
      ax += (double)fx;
      ay += (double)fy;
      az += (double)fz;
    }
  }
}

}  // namespace ladds
