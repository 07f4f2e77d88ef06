// propagate.hip -- Yoshida-4 propagation kernel (one thread per object).
//
// Replaces YoshidaIntegrator<AutoPas_t>::integrate (OrbitPropagator @ b90f3bae, called at
// src/ladds/Simulation.cpp:297).  One step is the 4th-order composition of Yoshida
// (Phys. Lett. A 150 (1990) 262):
//   r += c1 dt v; v += d1 dt a(r, v, t + c1 dt)
//   r += c2 dt v; v += d2 dt a(r, v, t + (c1+c2) dt)
//   r += c3 dt v; v += d3 dt a(r, v, t + (c1+c2+c3) dt)
//   r += c4 dt v
// with w1 = 1/(2 - 2^(1/3)), w0 = -2^(1/3)/(2 - 2^(1/3)), c1 = c4 = w1/2,
// c2 = c3 = (w0+w1)/2, d1 = d3 = w1, d2 = w0.  Velocity-dependent drag uses the
// latest kicked velocity; time-dependent terms use the sub-step time.
//
// Layout: SoA FP64 state in HBM, one coalesced 8-byte load/store per component.
// Several steps per launch keep the state in registers between steps (used when
// no conjunction scan is due in between).  When `count` is set, the kernel also
// performs the counting pass of the cell binning for the final positions.
#include <type_traits>

#include "binning.h"
#include "launch.h"
#include "physics.h"

namespace ladds {

__constant__ AtmTable c_atm;

struct PropagateArgs {
  DeviceObjects o;
  const SubstepEnv<double> *env64;  // 3 per step
  const SubstepEnv<float> *env32;
  int nsteps;
  unsigned mask;
  double cdt[4], ddt[3];
  GridParams grid;
  uint32_t *keys;   // non-null: write the bucket key of the binning point
  uint32_t *count;  // non-null: counting pass of the atomic counting sort
  uint32_t *slot;
  double burnup_r2;  // > 0: objects with |r|^2 below become dummies (deleteBurnUps)
  unsigned long long *burnups;  // non-null: count of objects flagged here
  const StepState *step_state;  // non-null (graph replay): environments start at step_state->step + step_offset
  uint32_t step_offset;
  // output state (the input arrays of `o` when propagating in place)
  double *orx, *ory, *orz, *ovx, *ovy, *ovz;
  int32_t *oact;
};

// STAGED: the environments go through LDS (EnvStage).  With one wavefront per SIMD or less the
// scalar loads of environments that no other wavefront of the XCD has read yet took half of
// a step (4,099 objects, FP64, components branched over: 3.83 us per step, 2.05 staged).
// With four (65,521 objects, ten steps a launch, 400 steps: 2.20 ms, 1.89 staged; 250,007, 1000
// steps: 6.14 and 5.97 ms) it still gains a little. Larger populations keep the 5.7 KB of LDS
// free for the pair kernel beside them (1,048,576 objects, split, 1,440 steps of the simulation
// loop: 95.4 ms staged, 94.0 without).
constexpr size_t kStagedObjects = 262144;

template <int FORM, bool STAGED>
__global__ __launch_bounds__(256) void k_propagate(PropagateArgs a) {
  __shared__ AtmTable atm;
  __shared__ EnvStage stage[STAGED ? 4 : 1][STAGED ? 2 : 1];
  {
    const double *src = reinterpret_cast<const double *>(&c_atm);
    double *dst = reinterpret_cast<double *>(&atm);
    for (int k = threadIdx.x; k < (int)(sizeof(AtmTable) / sizeof(double)); k += blockDim.x) dst[k] = src[k];
    __syncthreads();
  }
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool live = i < a.o.n;
  if (!STAGED && !live) return;
  const size_t env0 = a.step_state ? 3u * ((size_t)a.step_state->step + a.step_offset) : 0u;
  // lane l holds word l of the next step's environments
  const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
  auto fetch = [&](int s, double &d, double &f) {
    const size_t k = env0 + 3 * (size_t)s;
    if (lane < kEnvWords64) d = reinterpret_cast<const double *>(a.env64 + k)[lane];
    if (FORM != kFormFp64 && lane < kEnvWords32) f = reinterpret_cast<const double *>(a.env32 + k)[lane];
  };
  auto keep = [&](int s, double d, double f) {
    EnvStage &e = stage[w][s & 1];
    if (lane < kEnvWords64) reinterpret_cast<double *>(e.e64)[lane] = d;
    if (FORM != kFormFp64 && lane < kEnvWords32) reinterpret_cast<double *>(e.e32)[lane] = f;
    // the wavefront reads what its other lanes wrote: LDS operations of a wavefront stay in order
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  double next64 = 0.0, next32 = 0.0;
  if constexpr (STAGED) fetch(0, next64, next32);
  const size_t ii = live ? i : 0;  // lanes past the end only stage environments
  double x = a.o.rx[ii], y = a.o.ry[ii], z = a.o.rz[ii];
  double vx = a.o.vx[ii], vy = a.o.vy[ii], vz = a.o.vz[ii];
  ObjParams p;
  p.activity = a.o.activity[ii];
  p.drag64 = a.o.drag64[ii];
  if constexpr (FORM == kFormFp64) {
    p.srp64 = a.o.srp64[ii];
    p.srp32 = 0.f;
  } else {
    p.srp32 = a.o.srp32[ii];
    p.srp64 = 0.0;
  }
  if constexpr (STAGED) keep(0, next64, next32);
  // dummies (burnt-up objects awaiting compaction) keep their state
  bool moving = live && p.activity >= 0;
  bool burnt = false;
  // evasivePreserving objects feel the Keplerian term only (Particle.h:49-52)
  const unsigned mask = p.activity == 2 ? a.mask & kKepBit : a.mask;
  auto steps = [&](auto force) {
    for (int s = 0; s < a.nsteps; ++s) {
      if constexpr (STAGED) {
        if (s + 1 < a.nsteps) fetch(s + 1, next64, next32);
      }
      if (moving) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const double cdt = a.cdt[k], ddt = a.ddt[k];
          x = fma(cdt, vx, x);
          y = fma(cdt, vy, y);
          z = fma(cdt, vz, z);
          double ax, ay, az;
          if constexpr (STAGED)
            force(stage[w][s & 1].e64[k], stage[w][s & 1].e32[k], ax, ay, az);
          else
            force(a.env64[env0 + 3 * (size_t)s + k], a.env32[env0 + 3 * (size_t)s + k], ax, ay, az);
          vx = fma(ddt, ax, vx);
          vy = fma(ddt, ay, vy);
          vz = fma(ddt, az, vz);
        }
        x = fma(a.cdt[3], vx, x);
        y = fma(a.cdt[3], vy, y);
        z = fma(a.cdt[3], vz, z);
        // Simulation::deleteBurnUps after every integrate (Simulation.cpp:301-303, 589-590)
        if (a.burnup_r2 > 0.0 && exact_dot3(x, y, z, x, y, z) < a.burnup_r2) {
          burnt = true;
          moving = false;
        }
      }
      if constexpr (STAGED) {
        if (s + 1 < a.nsteps) keep(s + 1, next64, next32);
      }
    }
  };
  // The two usual models, without evasivePreserving objects in the wavefront, with a constant
  // mask: one block of straight code per kick, whose components' chains interleave (4,099
  // objects, full model, FP64: 2.05 -> 1.62 us per step; 1,048,576: 22.9 -> 20.3 us).  The path of all
  // others also takes objects beyond kFar (or not numbers).
  auto with = [&](unsigned m, auto far) {
    return [&, m](const SubstepEnv<double> &e64, const SubstepEnv<float> &e32, double &ax, double &ay, double &az) {
      acceleration<FORM, decltype(far)::value>(x, y, z, vx, vy, vz, p, m, e64, e32, atm, ax, ay, az);
    };
  };
  const unsigned long long usual = __ballot(mask != kAllBits), j2 = __ballot(mask != (kKepBit | kJ2Bit)),
                           far = __ballot(!(fabs(x) + fabs(y) + fabs(z) < kFar));
  if ((usual | far) == 0ull)
    steps(with(kAllBits, std::false_type{}));
  else if ((j2 | far) == 0ull)
    steps(with(kKepBit | kJ2Bit, std::false_type{}));
  else
    steps(with(mask, std::true_type{}));
  if (!live) return;
  if (burnt) {
    a.oact[i] = -1;
    if (a.burnups) atomicAdd(a.burnups, 1ull);  // rare: one atomic per burnt-up object
  }
  else if (a.oact != a.o.activity)
    a.oact[i] = p.activity;
  a.orx[i] = x;
  a.ory[i] = y;
  a.orz[i] = z;
  a.ovx[i] = vx;
  a.ovy[i] = vy;
  a.ovz[i] = vz;
  if (a.keys || a.count) {
    binning_point<FORM != kFormFp64>(x, y, z);
    const CellInfo c = cell_of(x, y, z, a.grid);
    if (a.keys)
      a.keys[i] = c.bucket;
    else
      a.slot[i] = atomicAdd(&a.count[c.bucket], 1u);
  }
}

template <int FORM>
void launch_propagate_as(const PropagateArgs &a, hipStream_t stream) {
  const dim3 blocks((unsigned)((a.o.n + 255) / 256)), threads(256);
  if (a.o.n <= kStagedObjects)
    hipLaunchKernelGGL((k_propagate<FORM, true>), blocks, threads, 0, stream, a);
  else
    hipLaunchKernelGGL((k_propagate<FORM, false>), blocks, threads, 0, stream, a);
}

hipError_t upload_atmosphere() {
  AtmTable t;
  fill_atm_table(t);
  return hipMemcpyToSymbol(HIP_SYMBOL(c_atm), &t, sizeof(t));
}

hipError_t launch_propagate(int form, const DeviceObjects &o, const SubstepEnv<double> *env64,
                            const SubstepEnv<float> *env32, int nsteps, unsigned mask, const double cdt[4],
                            const double ddt[3], const GridParams *grid, uint32_t *keys, uint32_t *count,
                            uint32_t *slot, double burnup_r2, const StepState *step_state, hipStream_t stream,
                            const DeviceObjects *out, uint32_t step_offset, unsigned long long *burnups) {
  if (o.n == 0 || nsteps <= 0) return hipSuccess;
  PropagateArgs a;
  a.o = o;
  const DeviceObjects &w = out ? *out : o;
  a.orx = w.rx;
  a.ory = w.ry;
  a.orz = w.rz;
  a.ovx = w.vx;
  a.ovy = w.vy;
  a.ovz = w.vz;
  a.oact = w.activity;
  a.env64 = env64;
  a.env32 = env32;
  a.nsteps = nsteps;
  a.mask = mask;
  for (int k = 0; k < 4; ++k) a.cdt[k] = cdt[k];
  for (int k = 0; k < 3; ++k) a.ddt[k] = ddt[k];
  if (grid) a.grid = *grid;
  a.keys = keys;
  a.count = count;
  a.slot = slot;
  a.burnup_r2 = burnup_r2;
  a.burnups = burnups;
  a.step_state = step_state;
  a.step_offset = step_offset;
  switch (form) {
    case kFormFp64:
      launch_propagate_as<kFormFp64>(a, stream);
      break;
    case kFormSplit:
      launch_propagate_as<kFormSplit>(a, stream);
      break;
    default:
      launch_propagate_as<kFormSplitAll32>(a, stream);
      break;
  }
  return hipGetLastError();
}

__global__ void k_set_step(StepState *st, uint32_t step, uint64_t iter_base) {
  if (threadIdx.x == 0) {
    st->step = step;
    st->pad = 0;
    st->iter_base = iter_base;
  }
}

__global__ void k_advance_step(StepState *st, uint32_t steps) {
  if (threadIdx.x == 0) st->step += steps;
}

hipError_t launch_set_step(StepState *st, uint32_t step, uint64_t iter_base, hipStream_t stream) {
  hipLaunchKernelGGL(k_set_step, dim3(1), dim3(64), 0, stream, st, step, iter_base);
  return hipGetLastError();
}

hipError_t launch_advance_step(StepState *st, uint32_t steps, hipStream_t stream) {
  hipLaunchKernelGGL(k_advance_step, dim3(1), dim3(64), 0, stream, st, steps);
  return hipGetLastError();
}

// Counters to the host: a kernel storing into coherent mapped host memory finishes a
// synchronised readback in ~11 us on MI355X, an 80-byte hipMemcpyAsync in ~21 us.
__global__ void k_publish(const unsigned long long *src, unsigned long long *dst, int words) {
  for (int k = threadIdx.x; k < words; k += blockDim.x) dst[k] = src[k];
}

// The same with the first entries of the pair log behind the counters: min(*log_count, `most`)
// entries of `entry_words` words each; *log_count (one of the published words) is reset.
__global__ void k_publish_log(const unsigned long long *src, unsigned long long *dst, int words,
                              unsigned long long *log_count, const unsigned long long *log,
                              unsigned long long *host_log, uint32_t most, uint32_t entry_words) {
  const unsigned long long cnt = *log_count;
  for (int k = threadIdx.x; k < words; k += blockDim.x) dst[k] = src[k];
  const uint32_t n = (cnt < most ? (uint32_t)cnt : most) * entry_words;
  for (uint32_t k = threadIdx.x; k < n; k += blockDim.x) host_log[k] = log[k];
  __syncthreads();  // every wavefront has read the count
  if (threadIdx.x == 0) *log_count = 0ull;
}

hipError_t launch_publish_log(const unsigned long long *src, unsigned long long *dst, int words,
                              unsigned long long *log_count, const LoggedPair *log, LoggedPair *host_log,
                              uint32_t most, hipStream_t stream) {
  static_assert(sizeof(LoggedPair) % 8 == 0, "whole words");
  hipLaunchKernelGGL(k_publish_log, dim3(1), dim3(256), 0, stream, src, dst, words, log_count,
                     reinterpret_cast<const unsigned long long *>(log),
                     reinterpret_cast<unsigned long long *>(host_log), most, (uint32_t)(sizeof(LoggedPair) / 8));
  return hipGetLastError();
}

hipError_t launch_publish(const unsigned long long *src, unsigned long long *dst, int words, hipStream_t stream) {
  hipLaunchKernelGGL(k_publish, dim3(1), dim3(64), 0, stream, src, dst, words);
  return hipGetLastError();
}

}  // namespace ladds
