// adjoint.hip -- hand-written adjoint of the FP64 Yoshida-4 propagation.
//
// Forward: the FP64 step of propagate.hip, every step of the trajectory in one launch, the state
// stored every K steps (checkpoints).  The force model stands here a second time, in four partial
// accelerations that also give their derivatives (partial_*, the same terms and constants as
// acceleration<kFormFp64>, fused and summed differently: the two agree to rounding).
//
// Backward: the gradient with respect to the initial state is a product of transition
// matrices, lambda_c = Phi_c^T lambda_{c+1}, one for each chunk of kChunk steps.  A chunk's
// matrix depends on its first state only, so chunks are independent: one thread per (object,
// checkpoint segment) recomputes the segment's steps from its checkpoint and carries the
// derivative of the state with respect to the chunk's first state (6 columns) and to bc_inv
// (a 7th) along,
//
//   step (v_k: velocity before kick k, r_k: position after drift k, h = dt)
//     r_k = r_{k-1} + c_k h v_k;   v_{k+1} = v_k + d_k h a(r_k, v_k, t_k)     k = 0, 1, 2
//     r'  = r_2 + c_3 h v_3;       v' = v_3
//   column (dr, dv):
//     dr += c_k h dv;              dv += d_k h (J_r dr + J_v dv  [+ da/dbc_inv])
//
// and a last launch applies the transposed matrices from the last chunk to the first.  Chunks
// begin at multiples of kChunk whatever the checkpoint spacing is, and forward and
// recomputation evaluate the same partial accelerations (contraction fixed by the source, summed
// in a fixed order), so the gradient does not depend on the spacing, to the last bit.  The
// reverse sweep this replaced (recompute a segment, then walk its steps back) was one chain
// of 8 force evaluations per step through the whole trajectory on 64 wavefronts.
//
// The Jacobians are derived by hand per component.  Every term except drag is the gradient
// of a potential (Kepler, J2, C22/S22 rotated with the Earth, the third bodies, cannonball
// SRP on the lit branch), so its part of J_r is a symmetric Hessian.  Drag
// a = D rho(h) |W| W with W = v - omega x r = v + B r, D = -1/2 1e3 bc_inv:
//   J_v = D rho (|W| I + W W^T/|W|)
//   J_r = W g^T + J_v B,   g = D |W| rho'(h) r/|r|,   B = ((0, omega, 0), (-omega, 0, 0), 0)
//   da/dbc_inv = -1/2 1e3 rho |W| W
// Branch decisions (shadow, atmosphere row) are those of the forward trajectory: the
// result is the derivative of the branch taken, as for any piecewise-smooth model.
//
// No LADDS counterpart: the reference has no differentiable propagation.  The forward
// matches YoshidaIntegrator::integrate (OrbitPropagator @ b90f3bae, Simulation.cpp:297).
#include <algorithm>
#include <cstring>
#include <string>
#include <vector>

#include "ephemeris.h"
#include "ladds_amd.h"
#include "physics.h"

namespace ladds {

__constant__ AtmTable c_atm_adj;

struct AdjointArgs {
  size_t n;
  int nsteps, every, nck;
  unsigned mask;
  double cdt[4], ddt[3];
  const SubstepEnv<double> *env;
  const double *aom, *bc, *cr;
  const int32_t *activity;
  const double *r0, *v0;  // [3][n]
  double *rT, *vT;        // [3][n]
  double *ck;             // [nck][6][n]
  const double *g_rT, *g_vT;
  double *g_r0, *g_v0, *g_bc;
  double *phi;            // transition matrices of chunks [chunk0, chunk0 + nchunk): [nchunk][kPhi][n]
  int chunk0, nchunk;
};

// Steps of one transition matrix: 32 make the matrices' traffic (336 bytes per object and
// chunk) small beside the recomputation, and cut 64-step segments in two.
constexpr int kChunk = 32;

// Entries of one transition matrix: 7 columns (initial position, initial velocity, bc_inv) of
// 6 rows (position, velocity).
constexpr int kPhi = 42;

__device__ __forceinline__ void stage_atm(AtmTable &atm) {
  const double *src = reinterpret_cast<const double *>(&c_atm_adj);
  double *dst = reinterpret_cast<double *>(&atm);
  for (int k = threadIdx.x; k < (int)(sizeof(AtmTable) / sizeof(double)); k += blockDim.x) dst[k] = src[k];
  __syncthreads();
}

__device__ __forceinline__ ObjParams object_params(const AdjointArgs &a, size_t i) {
  ObjParams p;
  const double aom = a.aom ? a.aom[i] : 0.0;
  const double cr = a.cr ? a.cr[i] : 1.0;
  const double bc = a.bc ? a.bc[i] : 0.0;
  p.srp64 = kSrpCoef * cr * aom;
  p.drag64 = kDragCoef * bc;
  p.srp32 = 0.f;
  p.activity = a.activity ? a.activity[i] : 0;
  return p;
}

struct State {
  double x, y, z, vx, vy, vz;
};

// Lane l's word of the environments of step s, and its store into the stage that the
// wavefront then reads (LDS operations of a wavefront stay in order).
__device__ __forceinline__ double fetch_env(const SubstepEnv<double> *env, int s, uint32_t lane) {
  return lane < kEnvWords64 ? reinterpret_cast<const double *>(env + 3 * (size_t)s)[lane] : 0.0;
}
__device__ __forceinline__ void keep_env(SubstepEnv<double> (&stage)[3], double word, uint32_t lane) {
  if (lane < kEnvWords64) reinterpret_cast<double *>(stage)[lane] = word;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// rsqrt64<true> with one instruction instead of three: scalar registers are free here (4,096 objects, a
// day of 60 s steps: 2.58 ms, 2.61 with the other).
__device__ __forceinline__ double rsqrt64_far(double x) {
  return rsqrt64_step(fmin(x, 1.7976931348623157e308), __builtin_amdgcn_rsq(x));
}

// Derivatives of the acceleration at (r, v).
struct Jacobian {
  double xx, xy, xz, yy, yz, zz;          // conservative part of da/dr (symmetric)
  double d[3][3];                         // drag's part of da/dr
  double vxx, vxy, vxz, vyy, vyz, vzz;    // da/dv (symmetric)
  double b[3];                            // da/dbc_inv
};

// The four partial accelerations, with their derivatives when LIN.

// Kepler, J2 and the tesseral terms: a = f r + (px, py, pz).
template <bool LIN>
__device__ __forceinline__ void partial_field(double x, double y, double z, unsigned mask, const SubstepEnv<double> &e,
                                              double (&a)[3], Jacobian &o) {
#pragma clang fp contract(on)
  const double r2 = x * x + y * y + z * z;
  const double inv_r = rsqrt64_far(r2);
  const double inv_r2 = inv_r * inv_r;
  const double inv_r3 = inv_r2 * inv_r;
  const double inv_r5 = inv_r3 * inv_r2;
  // da/dr = d I + c r r^T + what is added to o
  double f = 0.0, px = 0.0, py = 0.0, pz = 0.0, d = 0.0, c = 0.0;
  if (mask & kKepBit) {
    f = -kMuEarth * inv_r3;
    if (LIN) {
      d = f;
      c = 3.0 * kMuEarth * inv_r5;
    }
  }
  if (mask & kJ2Bit) {
    // a_i = fj x_i (c_i - z2), c = (1, 1, 3), fj = -kJ2Coef/r^5, z2 = 5 z^2/r^2:
    // da_i/dx_j = fj ((c_i - z2) delta_ij + x_i x_j/r^2 (7 z2 - 5 c_i) - 10 x_i z delta_jz/r^2)
    const double z2 = z * z * inv_r2 * 5.0;
    const double fj = -kJ2Coef * inv_r5;
    const double f1 = fj * (1.0 - z2);
    f += f1;
    pz = 2.0 * fj * z;
    if (LIN) {
      const double g = fj * inv_r2;
      const double gz = -10.0 * g * z;
      d += f1;
      c += g * (7.0 * z2 - 5.0);
      o.xz += gz * x;
      o.yz += gz * y;
      o.zz += 2.0 * fj + 2.0 * gz * z;
    }
  }
  if (mask & (kC22Bit | kS22Bit)) {
    // a = q/r^5 - 5 U r/r^7 with U = A (x^2 - y^2) + B x y, q = grad U
    double A, B;
    tesseral_coefficients(e, mask, A, B);
    const double U = A * ((x - y) * (x + y)) + B * (x * y);
    const double qx = 2.0 * A * x + B * y, qy = B * x - 2.0 * A * y;
    const double inv_r7 = inv_r5 * inv_r2;
    const double u5 = -5.0 * U * inv_r7;
    f += u5;
    px = qx * inv_r5;
    py = qy * inv_r5;
    if (LIN) {
      const double q5 = -5.0 * inv_r7;
      const double tx = q5 * qx, ty = q5 * qy;
      d += u5;
      c += -7.0 * u5 * inv_r2;
      o.xx += 2.0 * A * inv_r5 + 2.0 * tx * x;
      o.xy += B * inv_r5 + tx * y + ty * x;
      o.xz += tx * z;
      o.yy += 2.0 * ty * y - 2.0 * A * inv_r5;
      o.yz += ty * z;
    }
  }
  a[0] = fma(f, x, px);
  a[1] = fma(f, y, py);
  a[2] = fma(f, z, pz);
  if (LIN) {
    const double cx = c * x, cy = c * y, cz = c * z;
    o.xx += cx * x + d;
    o.xy += cx * y;
    o.xz += cx * z;
    o.yy += cy * y + d;
    o.yz += cy * z;
    o.zz += cz * z + d;
  }
}

// a = al W, al = D rho |W|.
template <bool LIN>
__device__ __forceinline__ void partial_drag(double x, double y, double z, double vx, double vy, double vz,
                                             double drag64, const AtmTable &atm, double (&a)[3], Jacobian &o) {
#pragma clang fp contract(on)
  const double om = kOmegaEarth;
  const double wx = vx + om * y, wy = vy - om * x, wz = vz;
  const double w2 = wx * wx + wy * wy + wz * wz;
  const double inv_w = rsqrt64<false>(fmax(w2, 1e-290));
  const double wn = w2 * inv_w;  // 0 without wind
  const double r2 = x * x + y * y + z * z;
  const double inv_r = rsqrt64_far(r2);
  const double h = r2 * inv_r - kREarth;
  const AtmRow &row = atm_row(h, atm);
  const double inv_scale = row.inv_scale;
  const double rho = row.rho * exp64((row.h0 - h) * inv_scale);
  const double dr = drag64 * rho;
  const double al = dr * wn;
  a[0] = al * wx;
  a[1] = al * wy;
  a[2] = al * wz;
  if (LIN) {
    const double s = dr * (w2 > 0.0 ? inv_w : 0.0);
    const double sx = s * wx, sy = s * wy, sz = s * wz;
    o.vxx = sx * wx + al;
    o.vxy = sx * wy;
    o.vxz = sx * wz;
    o.vyy = sy * wy + al;
    o.vyz = sy * wz;
    o.vzz = sz * wz + al;
    const double bw = kDragCoef * rho * wn;
    o.b[0] = bw * wx;
    o.b[1] = bw * wy;
    o.b[2] = bw * wz;
    const double gr = -al * inv_scale * inv_r;
    const double gx = gr * x, gy = gr * y, gz = gr * z;
    o.d[0][0] = wx * gx - om * o.vxy;
    o.d[0][1] = wx * gy + om * o.vxx;
    o.d[0][2] = wx * gz;
    o.d[1][0] = wy * gx - om * o.vyy;
    o.d[1][1] = wy * gy + om * o.vxy;
    o.d[1][2] = wy * gz;
    o.d[2][0] = wz * gx - om * o.vyz;
    o.d[2][1] = wz * gy + om * o.vxz;
    o.d[2][2] = wz * gz;
  }
}

// Central term k d/|d|^3, d = s - r, less the indirect term; its Hessian is
// -k/|d|^3 (I - 3 d d^T/|d|^2).
template <bool LIN>
__device__ __forceinline__ void partial_central(double x, double y, double z, const double *s, double k,
                                                const double *indirect, bool gravity, double (&a)[3], Jacobian &o) {
#pragma clang fp contract(on)
  const double dx = s[0] - x, dy = s[1] - y, dz = s[2] - z;
  const double inv_d = rsqrt64_far(dx * dx + dy * dy + dz * dz);
  const double inv_d2 = inv_d * inv_d;
  const double f = k * (inv_d2 * inv_d);
  const double go = gravity ? 1.0 : 0.0;
  a[0] = fma(f, dx, -go * indirect[0]);
  a[1] = fma(f, dy, -go * indirect[1]);
  a[2] = fma(f, dz, -go * indirect[2]);
  if (LIN) {
    const double c = 3.0 * f * inv_d2;
    const double cx = c * dx, cy = c * dy, cz = c * dz;
    o.xx += cx * dx - f;
    o.xy += cx * dy;
    o.xz += cx * dz;
    o.yy += cy * dy - f;
    o.yz += cy * dz;
    o.zz += cz * dz - f;
  }
}

// Partial acceleration `group` (0: Earth's field, 1: drag, 2: Sun and SRP, 3: Moon); zero
// where its components are off.
template <bool LIN>
__device__ __forceinline__ void partial_acceleration(int group, const State &s, const ObjParams &p, unsigned mask,
                                                     const SubstepEnv<double> &e, const AtmTable &atm,
                                                     double (&a)[3], Jacobian &o) {
#pragma clang fp contract(on)
  a[0] = a[1] = a[2] = 0.0;
  if (group == 0) {
    if (mask & (kKepBit | kJ2Bit | kC22Bit | kS22Bit)) partial_field<LIN>(s.x, s.y, s.z, mask, e, a, o);
  } else if (group == 1) {
    if (mask & kDragBit) partial_drag<LIN>(s.x, s.y, s.z, s.vx, s.vy, s.vz, p.drag64, atm, a, o);
  } else if (group == 2) {
    if (mask & (kSolBit | kSrpBit)) {
      double k = (mask & kSolBit) ? kGmSun : 0.0;
      const double r2 = s.x * s.x + s.y * s.y + s.z * s.z;
      if (mask & kSrpBit) k -= in_shadow(s.x, s.y, s.z, r2, e) ? 0.0 : p.srp64;
      partial_central<LIN>(s.x, s.y, s.z, e.sun, k, e.sun_acc, (mask & kSolBit) != 0, a, o);
    }
  } else {
    if (mask & kLunBit) partial_central<LIN>(s.x, s.y, s.z, e.moon, kGmMoon, e.moon_acc, true, a, o);
  }
}

// The sum of the four, in the order of the forward's exchange.
template <bool LIN>
__device__ __forceinline__ void total_acceleration(const State &s, const ObjParams &p, unsigned mask,
                                                   const SubstepEnv<double> &e, const AtmTable &atm, double (&a)[3],
                                                   Jacobian &o) {
  double b[3];
  partial_acceleration<LIN>(0, s, p, mask, e, atm, a, o);
#pragma unroll
  for (int g = 1; g < 4; ++g) {
    partial_acceleration<LIN>(g, s, p, mask, e, atm, b, o);
    for (int q = 0; q < 3; ++q) a[q] += b[q];
  }
}

// Drift and kick of the composition, contracted the same way everywhere.
__device__ __forceinline__ void drift(State &s, double cdt) {
  s.x = fma(cdt, s.vx, s.x);
  s.y = fma(cdt, s.vy, s.y);
  s.z = fma(cdt, s.vz, s.z);
}
__device__ __forceinline__ void kick(State &s, double ddt, const double (&a)[3]) {
  s.vx = fma(ddt, a[0], s.vx);
  s.vy = fma(ddt, a[1], s.vy);
  s.vz = fma(ddt, a[2], s.vz);
}

__device__ __forceinline__ void load_state(State &s, const double *base, size_t n, size_t i) {
  s.x = base[i];
  s.y = base[n + i];
  s.z = base[2 * n + i];
  s.vx = base[3 * n + i];
  s.vy = base[4 * n + i];
  s.vz = base[5 * n + i];
}

__device__ __forceinline__ void store_state(const State &s, double *base, size_t n, size_t i) {
  base[i] = s.x;
  base[n + i] = s.y;
  base[2 * n + i] = s.z;
  base[3 * n + i] = s.vx;
  base[4 * n + i] = s.vy;
  base[5 * n + i] = s.vz;
}

// The forward pass is one chain of steps.  Up to kGroupObjects objects (half a wavefront per
// SIMD at one thread per object) four wavefronts share 64 objects: wavefront w evaluates
// partial acceleration w, the four are summed through LDS, and every wavefront then carries
// the same integrator state.  With more objects one thread per object fills the SIMDs without
// the exchange.
constexpr int kAdjWaves = 4;
constexpr int kAdjLanes = 64;
constexpr size_t kGroupObjects = 32768;

// Dummies keep their state; evasivePreserving objects feel the Keplerian term only.
__device__ __forceinline__ unsigned object_mask(const ObjParams &p, unsigned mask) {
  return p.activity == 2 ? mask & kKepBit : mask;
}

template <bool GROUPED>
__global__ __launch_bounds__(kAdjWaves *kAdjLanes) void k_adjoint_forward(AdjointArgs a) {
  __shared__ AtmTable atm;
  // partial sums of the four wavefronts, double-buffered: one barrier per exchange, since a
  // buffer is rewritten only after the next exchange's barrier, which every wavefront reaches
  // after reading it
  __shared__ double part[GROUPED ? 2 : 1][GROUPED ? kAdjWaves : 1][3][kAdjLanes];
  __shared__ SubstepEnv<double> stage[kAdjWaves][2][3];
  stage_atm(atm);
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kAdjLanes));
  const uint32_t l = threadIdx.x % kAdjLanes;
  const size_t n = a.n, i = (GROUPED ? (size_t)blockIdx.x : (size_t)blockIdx.x * kAdjWaves + w) * kAdjLanes + l;
  const bool live = i < n;
  const size_t ii = live ? i : 0;  // lanes past the end compute on object 0 and write nothing
  const bool writes = live && (!GROUPED || w == 0);
  State s{a.r0[ii], a.r0[n + ii], a.r0[2 * n + ii], a.v0[ii], a.v0[n + ii], a.v0[2 * n + ii]};
  const ObjParams p = object_params(a, ii);
  const unsigned mask = object_mask(p, a.mask);
  const bool moving = p.activity >= 0;
  Jacobian unused;
  int parity = 0, until = 0;  // until: steps to the next checkpoint
  double next = fetch_env(a.env, 0, l);
  keep_env(stage[w][0], next, l);
  double *ck = a.ck;
  for (int step = 0; step < a.nsteps; ++step) {
    if (until == 0) {
      if (writes) store_state(s, ck, n, i);
      ck += 6 * n;
      until = a.every;
    }
    until -= 1;
    if (step + 1 < a.nsteps) next = fetch_env(a.env, step + 1, l);
    const SubstepEnv<double> *env = stage[w][step & 1];
    State t = s;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      drift(t, a.cdt[k]);
      double acc[3];
      if constexpr (GROUPED) {
        partial_acceleration<false>(w, t, p, mask, env[k], atm, acc, unused);
        for (int q = 0; q < 3; ++q) part[parity][w][q][l] = acc[q];
        __syncthreads();
        for (int q = 0; q < 3; ++q)
          acc[q] = ((part[parity][0][q][l] + part[parity][1][q][l]) + part[parity][2][q][l]) + part[parity][3][q][l];
        parity ^= 1;
      } else {
        total_acceleration<false>(t, p, mask, env[k], atm, acc, unused);
      }
      kick(t, a.ddt[k], acc);
    }
    drift(t, a.cdt[3]);
    if (moving) s = t;
    if (step + 1 < a.nsteps) keep_env(stage[w][(step + 1) & 1], next, l);
  }
  if (writes) {
    a.rT[i] = s.x;
    a.rT[n + i] = s.y;
    a.rT[2 * n + i] = s.z;
    a.vT[i] = s.vx;
    a.vT[n + i] = s.vy;
    a.vT[2 * n + i] = s.vz;
  }
}

// Transition matrices for 64 objects: of the chunks of [a.chunk0, a.chunk0 + a.nchunk) that
// begin in one checkpoint segment, or (segments shorter than a chunk) of one chunk.
__global__ __launch_bounds__(kAdjLanes) __attribute__((amdgpu_waves_per_eu(2)))
void k_adjoint_segments(AdjointArgs a) {
  __shared__ AtmTable atm;
  __shared__ SubstepEnv<double> stage[2][3];
  stage_atm(atm);
  const uint32_t l = threadIdx.x;
  const size_t n = a.n, i = (size_t)blockIdx.x * kAdjLanes + l;
  const bool live = i < n;
  const size_t ii = live ? i : 0;
  int seg, first, last;  // chunks [first, last) from the checkpoint of segment seg
  if (a.every < kChunk) {
    first = a.chunk0 + (int)blockIdx.y;
    last = first + 1;
    seg = first * kChunk / a.every;
  } else {
    seg = a.chunk0 * kChunk / a.every + (int)blockIdx.y;
    first = max(a.chunk0, (seg * a.every + kChunk - 1) / kChunk);
    last = min(a.chunk0 + a.nchunk, (min((seg + 1) * a.every, a.nsteps) + kChunk - 1) / kChunk);
  }
  if (first >= last) return;
  State s;
  load_state(s, a.ck + (size_t)seg * 6 * n, n, ii);
  const ObjParams p = object_params(a, ii);
  const unsigned mask = object_mask(p, a.mask);
  int step = seg * a.every;
  const int end = min(last * kChunk, a.nsteps);
  double next = fetch_env(a.env, step, l);
  keep_env(stage[step & 1], next, l);
  // to the first chunk
  for (; step < first * kChunk; ++step) {
    next = fetch_env(a.env, step + 1, l);
#pragma unroll 1
    for (int k = 0; k < 3; ++k) {
      drift(s, a.cdt[k]);
      double acc[3];
      Jacobian unused;
      total_acceleration<false>(s, p, mask, stage[step & 1][k], atm, acc, unused);
      kick(s, a.ddt[k], acc);
    }
    drift(s, a.cdt[3]);
    keep_env(stage[(step + 1) & 1], next, l);
  }
  double R[7][3], V[7][3];
#pragma unroll 1
  for (int chunk = first; chunk < last; ++chunk) {
#pragma unroll
    for (int c = 0; c < 7; ++c)
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        R[c][q] = c == q ? 1.0 : 0.0;
        V[c][q] = c == q + 3 ? 1.0 : 0.0;
      }
    const int stop = min((chunk + 1) * kChunk, a.nsteps);
#pragma unroll 1
    for (; step < stop; ++step) {
      if (step + 1 < end) next = fetch_env(a.env, step + 1, l);
#pragma unroll 1
      for (int k = 0; k < 3; ++k) {
        const double cdt = a.cdt[k], ddt = a.ddt[k];
        drift(s, cdt);
        Jacobian j{};
        double acc[3];
        total_acceleration<true>(s, p, mask, stage[step & 1][k], atm, acc, j);
        kick(s, ddt, acc);
        const double xx = ddt * (j.xx + j.d[0][0]), xy = ddt * (j.xy + j.d[0][1]), xz = ddt * (j.xz + j.d[0][2]);
        const double yx = ddt * (j.xy + j.d[1][0]), yy = ddt * (j.yy + j.d[1][1]), yz = ddt * (j.yz + j.d[1][2]);
        const double zx = ddt * (j.xz + j.d[2][0]), zy = ddt * (j.yz + j.d[2][1]), zz = ddt * (j.zz + j.d[2][2]);
        const double vxx = ddt * j.vxx, vxy = ddt * j.vxy, vxz = ddt * j.vxz, vyy = ddt * j.vyy, vyz = ddt * j.vyz,
                     vzz = ddt * j.vzz;
#pragma unroll
        for (int c = 0; c < 7; ++c) {
          const double ux = V[c][0], uy = V[c][1], uz = V[c][2];
          const double rx = R[c][0] += cdt * ux, ry = R[c][1] += cdt * uy, rz = R[c][2] += cdt * uz;
          V[c][0] += xx * rx + xy * ry + xz * rz + vxx * ux + vxy * uy + vxz * uz;
          V[c][1] += yx * rx + yy * ry + yz * rz + vxy * ux + vyy * uy + vyz * uz;
          V[c][2] += zx * rx + zy * ry + zz * rz + vxz * ux + vyz * uy + vzz * uz;
        }
#pragma unroll
        for (int q = 0; q < 3; ++q) V[6][q] += ddt * j.b[q];
      }
      const double cdt = a.cdt[3];
      drift(s, cdt);
#pragma unroll
      for (int c = 0; c < 7; ++c)
#pragma unroll
        for (int q = 0; q < 3; ++q) R[c][q] += cdt * V[c][q];
      if (step + 1 < end) keep_env(stage[(step + 1) & 1], next, l);
    }
    if (live) {
      double *out = a.phi + (size_t)(chunk - a.chunk0) * kPhi * n + i;
#pragma unroll
      for (int c = 0; c < 7; ++c)
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          out[(size_t)(6 * c + q) * n] = R[c][q];
          out[(size_t)(6 * c + 3 + q) * n] = V[c][q];
        }
    }
  }
}

// lambda = Phi^T lambda over the chunks [chunk0, chunk0 + nchunk), last to first.  The first
// call (the trajectory's last chunks) starts from the loss gradient, the later ones from what
// the previous call left in the outputs.
__global__ __launch_bounds__(kAdjLanes) void k_adjoint_chain(AdjointArgs a) {
  const size_t n = a.n, i = (size_t)blockIdx.x * kAdjLanes + threadIdx.x;
  if (i >= n) return;
  const bool first = (a.chunk0 + a.nchunk) * kChunk >= a.nsteps;
  const double *sr = first ? a.g_rT : a.g_r0, *sv = first ? a.g_vT : a.g_v0;
  double g[6];
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    g[q] = sr ? sr[q * n + i] : 0.0;
    g[3 + q] = sv ? sv[q * n + i] : 0.0;
  }
  double gbc = (!first && a.g_bc) ? a.g_bc[i] : 0.0;
  // dummies: no gradient flows through a deleted object
  const bool moving = !a.activity || a.activity[i] >= 0;
  // Three matrices in registers: two are on their way while one is applied (a wavefront per CU, so
  // nothing else hides their reads; 4,096 objects, 45 chunks: 207 -> 24 us).
  double v[3][kPhi];
  auto load = [&](double (&m)[kPhi], int c) {
    const double *p = a.phi + (size_t)c * kPhi * n + i;
#pragma unroll
    for (int q = 0; q < kPhi; ++q) m[q] = p[(size_t)q * n];
  };
  const int last = moving ? a.nchunk - 1 : -1;
  if (last >= 0) load(v[0], last);
  if (last >= 1) load(v[1], last - 1);
#pragma unroll 1
  for (int c0 = last; c0 >= 0; c0 -= 3) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int c = c0 - k;
      if (c < 0) break;
      if (c >= 2) load(v[(k + 2) % 3], c - 2);
      const double (&m)[kPhi] = v[k];
      double h[7];
#pragma unroll
      for (int j = 0; j < 7; ++j)
        h[j] = ((m[6 * j] * g[0] + m[6 * j + 1] * g[1]) + m[6 * j + 2] * g[2]) +
               ((m[6 * j + 3] * g[3] + m[6 * j + 4] * g[4]) + m[6 * j + 5] * g[5]);
#pragma unroll
      for (int q = 0; q < 6; ++q) g[q] = h[q];
      gbc += h[6];
    }
  }
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    a.g_r0[q * n + i] = g[q];
    a.g_v0[q * n + i] = g[3 + q];
  }
  if (a.g_bc) a.g_bc[i] = gbc;
}

}  // namespace ladds

using namespace ladds;

struct ladds_adjoint {
  ladds_adjoint_config cfg{};
  int every = 64, nck = 0;
  std::string err;
  SubstepEnv<double> *env = nullptr;
  double *phi = nullptr;  // transition matrices of `group` chunks
  int group = 1;
  double cdt[4], ddt[3];
  int fail(int code, const std::string &m) {
    err = m;
    return code;
  }
  int hipfail(hipError_t e, const char *what) {
    err = std::string(what) + ": " + hipGetErrorString(e);
    return e == hipErrorOutOfMemory ? LADDS_E_NOMEM : LADDS_E_HIP;
  }
};

#define ADJCHK(p, call)                                   \
  do {                                                    \
    hipError_t e_ = (call);                               \
    if (e_ != hipSuccess) return (p)->hipfail(e_, #call); \
  } while (0)

extern "C" {

int ladds_adjoint_create(const ladds_adjoint_config *cfg, ladds_adjoint **out) {
  if (!cfg || !out || cfg->n == 0 || cfg->nsteps < 1 || cfg->checkpoint_every < 0 || !(cfg->dt > 0.0))
    return LADDS_E_INVALID;
  *out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || cfg->device < 0 || cfg->device >= ndev) return LADDS_E_NODEVICE;
  auto *p = new ladds_adjoint;
  p->cfg = *cfg;
  p->every = cfg->checkpoint_every > 0 ? cfg->checkpoint_every : 64;
  if (p->every > cfg->nsteps) p->every = cfg->nsteps;
  p->nck = (cfg->nsteps + p->every - 1) / p->every;
  double c[4], d[3];
  yoshida_coefficients(c, d);
  for (int k = 0; k < 4; ++k) p->cdt[k] = c[k] * cfg->dt;
  for (int k = 0; k < 3; ++k) p->ddt[k] = d[k] * cfg->dt;
  const double tau[3] = {c[0], c[0] + c[1], c[0] + c[1] + c[2]};
  std::vector<SubstepEnv<double>> env(3 * (size_t)cfg->nsteps);
  for (int s = 0; s < cfg->nsteps; ++s) {
    const double t = cfg->t0 + (double)s * cfg->dt;
    for (int k = 0; k < 3; ++k) {
      SubstepEnv<float> e32;
      substep_env(t + tau[k] * cfg->dt, env[3 * s + k], e32);
    }
  }
  hipError_t e = hipSetDevice(cfg->device);
  AtmTable t;
  fill_atm_table(t);
  if (e == hipSuccess) e = hipMemcpyToSymbol(HIP_SYMBOL(c_atm_adj), &t, sizeof(t));
  if (e == hipSuccess) e = hipMalloc(&p->env, sizeof(SubstepEnv<double>) * env.size());
  if (e == hipSuccess) e = hipMemcpy(p->env, env.data(), sizeof(SubstepEnv<double>) * env.size(), hipMemcpyHostToDevice);
  // Matrices of as many chunks at once as 256 MiB hold, or what one segment's states would take
  // if that is more; at most 1,024 (a grid dimension holds 65,535 segments)
  const size_t chunk_bytes = sizeof(double) * kPhi * cfg->n, chunks = ((size_t)cfg->nsteps + kChunk - 1) / kChunk;
  const size_t budget = std::max<size_t>((size_t)256 << 20, sizeof(double) * 6 * cfg->n * (size_t)p->every);
  p->group = (int)std::min<size_t>({chunks, std::max<size_t>(1, budget / chunk_bytes), 1024});
  if (e == hipSuccess) e = hipMalloc(&p->phi, chunk_bytes * (size_t)p->group);
  if (e != hipSuccess) {
    hipFree(p->env);
    hipFree(p->phi);
    delete p;
    return e == hipErrorOutOfMemory ? LADDS_E_NOMEM : LADDS_E_HIP;
  }
  *out = p;
  return LADDS_OK;
}

int ladds_adjoint_destroy(ladds_adjoint *p) {
  if (!p) return LADDS_E_INVALID;
  (void)hipSetDevice(p->cfg.device);
  hipFree(p->env);
  hipFree(p->phi);
  delete p;
  return LADDS_OK;
}

const char *ladds_adjoint_last_error(const ladds_adjoint *p) { return p ? p->err.c_str() : "null plan"; }

uint64_t ladds_adjoint_checkpoint_doubles(const ladds_adjoint *p) {
  return p ? (uint64_t)p->nck * 6u * p->cfg.n : 0u;
}

static AdjointArgs make_args(const ladds_adjoint *p) {
  AdjointArgs a{};
  a.n = p->cfg.n;
  a.nsteps = p->cfg.nsteps;
  a.every = p->every;
  a.nck = p->nck;
  a.mask = p->cfg.components;
  for (int k = 0; k < 4; ++k) a.cdt[k] = p->cdt[k];
  for (int k = 0; k < 3; ++k) a.ddt[k] = p->ddt[k];
  a.env = p->env;
  a.phi = p->phi;
  return a;
}

int ladds_adjoint_forward(ladds_adjoint *p, const double *r0, const double *v0, const double *aom,
                          const double *bc_inv, const double *cr, const int32_t *activity, double *rT, double *vT,
                          double *checkpoints, void *stream) {
  if (!p) return LADDS_E_INVALID;
  if (!r0 || !v0 || !rT || !vT || !checkpoints) return p->fail(LADDS_E_INVALID, "null state or checkpoint pointer");
  ADJCHK(p, hipSetDevice(p->cfg.device));
  AdjointArgs a = make_args(p);
  a.aom = aom;
  a.bc = bc_inv;
  a.cr = cr;
  a.activity = activity;
  a.r0 = r0;
  a.v0 = v0;
  a.rT = rT;
  a.vT = vT;
  a.ck = checkpoints;
  const bool grouped = a.n <= kGroupObjects;
  const size_t per_block = grouped ? kAdjLanes : kAdjWaves * kAdjLanes;
  const dim3 blocks((unsigned)((a.n + per_block - 1) / per_block)), threads(kAdjWaves * kAdjLanes);
  if (grouped)
    hipLaunchKernelGGL(k_adjoint_forward<true>, blocks, threads, 0, (hipStream_t)stream, a);
  else
    hipLaunchKernelGGL(k_adjoint_forward<false>, blocks, threads, 0, (hipStream_t)stream, a);
  ADJCHK(p, hipGetLastError());
  return LADDS_OK;
}

int ladds_adjoint_backward(ladds_adjoint *p, const double *aom, const double *bc_inv, const double *cr,
                           const int32_t *activity, const double *checkpoints, const double *g_rT,
                           const double *g_vT, double *g_r0, double *g_v0, double *g_bc, void *stream) {
  if (!p) return LADDS_E_INVALID;
  if (!checkpoints || !g_r0 || !g_v0) return p->fail(LADDS_E_INVALID, "null checkpoint or gradient pointer");
  ADJCHK(p, hipSetDevice(p->cfg.device));
  AdjointArgs a = make_args(p);
  a.aom = aom;
  a.bc = bc_inv;
  a.cr = cr;
  a.activity = activity;
  a.ck = const_cast<double *>(checkpoints);
  a.g_rT = g_rT;
  a.g_vT = g_vT;
  a.g_r0 = g_r0;
  a.g_v0 = g_v0;
  a.g_bc = g_bc;
  const unsigned blocks = (unsigned)((a.n + kAdjLanes - 1) / kAdjLanes);
  const int chunks = (a.nsteps + kChunk - 1) / kChunk;
  for (int end = chunks; end > 0; end -= p->group) {
    a.chunk0 = std::max(0, end - p->group);
    a.nchunk = end - a.chunk0;
    // chunks that begin in one segment are one thread's
    const int runs = a.every < kChunk ? a.nchunk : (end - 1) * kChunk / a.every - a.chunk0 * kChunk / a.every + 1;
    hipLaunchKernelGGL(k_adjoint_segments, dim3(blocks, (unsigned)runs), dim3(kAdjLanes), 0, (hipStream_t)stream, a);
    ADJCHK(p, hipGetLastError());
    hipLaunchKernelGGL(k_adjoint_chain, dim3(blocks), dim3(kAdjLanes), 0, (hipStream_t)stream, a);
    ADJCHK(p, hipGetLastError());
  }
  return LADDS_OK;
}

}  // extern "C"
