// CartPole on MI355X: the single-step kernel, the K-step fused kernel, the
// reset kernel and the device action sampler, plus their C-ABI entry points.
//
// One thread per environment, state in VGPRs, SoA fp32 rows (x, x_dot, theta,
// theta_dot; row r of env i at r * n + i) so every access is coalesced. The physics is
// Gym's CartPole-v1 Euler step in the operation order of cartpole_np.py:58-76,
// termination cartpole_np.py:79-83, masked reset from the counter RNG exactly
// as cartpole_metal.py:84-95 writes it. Per env-step the single-step kernel
// moves 41 algorithmic bytes: 16 B state in, 4 B action, 16 B state out,
// 4 B reward, 1 B done.

#include "es_rollout.h"

namespace hipenvs {
namespace cp {

constexpr float GRAVITY = 0x1.39999ap+3f;           // float32(9.8)
constexpr float POLE_MASS = 0x1.99999ap-4f;         // float32(0.1)
constexpr float TOTAL_MASS = 0x1.19999ap+0f;        // float32(1.0 + 0.1)
constexpr float HALF_POLE_LENGTH = 0x1p-1f;         // float32(0.5)
constexpr float POLE_MASS_LENGTH = 0x1.99999ap-5f;  // float32(0.1 * 0.5)
constexpr float FORCE_MAG = 0x1.4p+3f;              // float32(10.0)
constexpr float TAU = 0x1.47ae14p-6f;               // float32(0.02)
constexpr float FOUR_THIRDS = 0x1.555556p+0f;       // float32(4.0 / 3.0)
constexpr float X_LIMIT = 0x1.333334p+1f;           // float32(2.4)
constexpr float THETA_LIMIT = 0x1.aceeap-3f;        // float32(12 * 2 * pi / 360)
constexpr float RESET_BOUND = 0x1.99999ap-5f;       // float32(0.05)
constexpr double INV_TOTAL_MASS = 1.0 / (double)TOTAL_MASS;  // for div_const(x, .) == x / TOTAL_MASS

// One explicit-Euler step in place; returns the termination flag.
// cartpole_np.py:58-83, each line evaluated in numpy's order.
// `exact` false marks a lane whose results are discarded (see det_sincos_near_zero).
__device__ __forceinline__ bool advance(float& x, float& xd, float& th, float& thd, int32_t action,
                                        bool exact = true) {
  const float force = (action == 1) ? FORCE_MAG : -FORCE_MAG;
  float s, c;
  det_sincos_near_zero(th, &s, &c, exact);  // the pole angle stays within +-0.78 but for a terminating step
  const float temp = div_const(force + (POLE_MASS_LENGTH * (thd * thd)) * s, INV_TOTAL_MASS);
  const float theta_acc = (GRAVITY * s - c * temp) /
                          (HALF_POLE_LENGTH * (FOUR_THIRDS - div_const(POLE_MASS * (c * c), INV_TOTAL_MASS)));
  const float x_acc = temp - div_const((POLE_MASS_LENGTH * theta_acc) * c, INV_TOTAL_MASS);
  x = x + TAU * xd;
  xd = xd + TAU * x_acc;
  th = th + TAU * thd;
  thd = thd + TAU * theta_acc;
  return (fabsf(x) > X_LIMIT) || (fabsf(th) > THETA_LIMIT);
}

// Masked reset (cartpole_metal.py:86-93): a terminated env takes four fresh draws. The
// reference computes the draws for every env and selects; here they sit on the branch of
// the terminated lanes, so a wave in which no env terminates skips the four hashes.
__device__ __forceinline__ void reset_select(bool d, uint32_t h, float& x, float& xd, float& th, float& thd) {
  if (d) {
    x = uniform_pm(pcg_hash(h), RESET_BOUND);
    xd = uniform_pm(pcg_hash(h + kRowOff1), RESET_BOUND);
    th = uniform_pm(pcg_hash(h + kRowOff2), RESET_BOUND);
    thd = uniform_pm(pcg_hash(h + kRowOff3), RESET_BOUND);
  }
}

// ---- kernels ---------------------------------------------------------------

__global__ __launch_bounds__(kBlock) void reset_kernel(float* __restrict__ state, uint32_t seed, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  float x = 0.f, xd = 0.f, th = 0.f, thd = 0.f;
  reset_select(true, env_hash(seed, (uint32_t)i), x, xd, th, thd);
  state[i] = x;
  state[n + i] = xd;
  state[2 * n + i] = th;
  state[3 * n + i] = thd;
}

// One env per thread, any n and alignment. At every batch size this beats packing four
// envs per thread into 16-byte accesses (2.96 vs 3.81 us at N = 2^18, 7.9 vs 9.3 us at
// 2^20): a step is short, and the extra waves hide more of the load latency.
// The four reset draws depend only on the seed and the env index, so they are computed
// for every env (as the reference's select does) while its state loads are in flight;
// the empty asm marks the draws as needed there, which keeps the compiler from sinking
// them past the physics, where they would add to the step's latency instead.
__global__ __launch_bounds__(kBlock) void step_kernel(const float* __restrict__ state, const int32_t* __restrict__ action,
                                                      uint32_t seed, float* __restrict__ next, float* __restrict__ reward,
                                                      uint8_t* __restrict__ done, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  float x = state[i], xd = state[n + i], th = state[2 * n + i], thd = state[3 * n + i];
  const int32_t a = stream_load(action + i);
  const uint32_t h = env_hash(seed, (uint32_t)i);
  float f0 = uniform_pm(pcg_hash(h), RESET_BOUND);
  float f1 = uniform_pm(pcg_hash(h + kRowOff1), RESET_BOUND);
  float f2 = uniform_pm(pcg_hash(h + kRowOff2), RESET_BOUND);
  float f3 = uniform_pm(pcg_hash(h + kRowOff3), RESET_BOUND);
  asm volatile("" : "+v"(f0), "+v"(f1), "+v"(f2), "+v"(f3));
  const bool d = advance(x, xd, th, thd, a);
  next[i] = d ? f0 : x;
  next[n + i] = d ? f1 : xd;
  next[2 * n + i] = d ? f2 : th;
  next[3 * n + i] = d ? f3 : thd;
  stream_store(1.0f, reward + i);
  stream_store((uint8_t)(d ? 1 : 0), done + i);
}

// k chained steps, one env per thread (any n): rewards and dones written per step as
// (k, n) rows, the state once at the end. One env per thread also wins here over four
// per thread (31.9 vs 44.3 us for k = 32 at N = 2^18): the loop is VALU-bound and more
// waves per SIMD keep the issue slots full.
template <bool kArrayActions>
__global__ __launch_bounds__(kBlock) void step_k_kernel(const float* __restrict__ state, const int32_t* __restrict__ actions,
                                                        uint32_t seed, int32_t k, float* __restrict__ next,
                                                        float* __restrict__ rewards, uint8_t* __restrict__ dones, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  float x = state[i], xd = state[n + i], th = state[2 * n + i], thd = state[3 * n + i];
  for (int32_t t = 0; t < k; ++t) {
    const uint32_t h = env_hash(seed + (uint32_t)t, (uint32_t)i);
    const int32_t a = kArrayActions ? stream_load(actions + (int64_t)t * n + i) : action_bit(h);
    const bool d = advance(x, xd, th, thd, a);
    reset_select(d, h, x, xd, th, thd);
    stream_store(1.0f, rewards + (int64_t)t * n + i);
    stream_store((uint8_t)(d ? 1 : 0), dones + (int64_t)t * n + i);
  }
  next[i] = x;
  next[n + i] = xd;
  next[2 * n + i] = th;
  next[3 * n + i] = thd;
}

__global__ __launch_bounds__(kBlock) void sample_actions_kernel(int32_t* __restrict__ action, int64_t n, uint32_t m,
                                                                uint32_t seed) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const uint32_t h = env_hash(seed, (uint32_t)i);
  action[i] = (m == 2u) ? action_bit(h) : action_uniform(h, m);
}

// The fused ES rollout's body (es_rollout.h): the 4-H-2 tanh policy with first-index argmax and
// the step physics; a member's score is the steps survived, the terminating step not counted
// (cartpole_rollout_metal.py:46-77).
struct RolloutBody {
  static constexpr int kIn = 4, kOut = 2;
  // the one-lane form keeps all 7H + 2 weights in registers: two waves per SIMD at H = 32
  template <int H, int G>
  static constexpr int kMinWaves = (G == 1 && H == 32) ? 2 : 1;
  struct Trig {};
  template <int G>
  __device__ static __forceinline__ Trig trig(const roll::State4&, int) {
    return {};
  }
  __device__ static __forceinline__ void observe(const roll::State4& s, const Trig&, float (&obs)[4]) {
    obs[0] = s.a;
    obs[1] = s.b;
    obs[2] = s.c;
    obs[3] = s.d;
  }
  // every member steps (no branch around the physics); the near-zero sin/cos vote counts the
  // live members alone, since a finished member's results are discarded
  template <int G>
  __device__ static __forceinline__ bool step(roll::State4& s, Trig&, const float (&l)[2], bool alive, int) {
    return advance(s.a, s.b, s.c, s.d, (l[1] > l[0]) ? 1 : 0, alive);
  }
  // steps as a float32 count that stops at 2^24, where adding one no longer changes it
  __device__ static __forceinline__ float score(int32_t t, float) { return (float)(t < 0x1000000 ? t : 0x1000000); }
};

// Lanes per member at the start, by members per CU. Trained populations (every member runs
// the 500 steps, P on 256 CUs, us; 16 / 4 / 1 lanes):
//   H = 32: P = 4,096 293 / 489 / 1,379; 8,192 356 / 530 / 1,383; 32,768 1,002 / 819 / 1,413;
//           65,536 1,816 / 1,294 / 1,416; 262,144 6,689 / 4,387 / 4,133
//   H = 8:  P = 8,192 240 / 264 / 446; 32,768 631 / 296 / 469; 65,536 1,089 / 456 / 449
//   H = 64: P = 8,192 563 / 916; 65,536 3,153 / 2,378 (its 450 weights leave one lane one wave
//           per SIMD: 2,864)
// Populations early in training, whose waves narrow as their members fail, are within 10 %
// between the forms at these bounds. One member per lane to the end, with the same arithmetic,
// takes 3,899 us at P = 262,144, H = 32 early in training and 3,891 trained, this kernel 574 and
// 4,135: the check for finished members and the registers of the other forms cost a population
// that runs to the horizon 6 %.
constexpr int kGroup16PerCu = 32;
template <int H>
constexpr int kGroup4PerCu = H >= 16 ? 256 : 128;

template <int H>
int launch_rollout(const float* state, const float* theta, int64_t member_stride, int64_t p, int32_t horizon,
                   float* out, hipStream_t s) {
  int cus = 0;
  const int status = device_cus(&cus);
  if (status != HIPENVS_OK) return status;
  if (p <= (int64_t)kGroup16PerCu * cus)
    return roll::launch<RolloutBody, H, 16>(state, theta, member_stride, p, horizon, 1.0f, out, s);
  if (H > 32 || p <= (int64_t)kGroup4PerCu<H> * cus)
    return roll::launch<RolloutBody, H, 4>(state, theta, member_stride, p, horizon, 1.0f, out, s);
  return roll::launch<RolloutBody, H, (H > 32 ? 4 : 1)>(state, theta, member_stride, p, horizon, 1.0f, out, s);
}

template <int H>
int launch_rollout(const float* state, const float* theta, int64_t p, int32_t horizon, float* out, hipStream_t s) {
  return launch_rollout<H>(state, theta, (int64_t)(7 * H + 2), p, horizon, out, s);
}

}  // namespace cp
}  // namespace hipenvs

using namespace hipenvs;

extern "C" int hipenvs_cartpole_reset(float* state, int64_t n, uint32_t seed, hipenvs_stream_t stream) {
  if (n < 0 || (n > 0 && !state)) return HIPENVS_E_ARG;
  if (n == 0) return HIPENVS_OK;
  hipLaunchKernelGGL(cp::reset_kernel, dim3(grid_for(n)), dim3(kBlock), 0, as_stream(stream), state, seed, n);
  return launch_status();
}

extern "C" int hipenvs_cartpole_step(const float* state, const int32_t* action, uint32_t seed, float* next_state,
                                     float* reward, uint8_t* done, int64_t n, hipenvs_stream_t stream) {
  if (n < 0 || (n > 0 && (!state || !action || !next_state || !reward || !done))) return HIPENVS_E_ARG;
  if (n == 0) return HIPENVS_OK;
  hipLaunchKernelGGL(cp::step_kernel, dim3(grid_for(n)), dim3(kBlock), 0, as_stream(stream), state, action, seed,
                     next_state, reward, done, n);
  return launch_status();
}

extern "C" int hipenvs_cartpole_step_k(const float* state, const int32_t* actions, uint32_t seed, int32_t k,
                                       float* next_state, float* rewards, uint8_t* dones, int64_t n,
                                       hipenvs_stream_t stream) {
  if (n < 0 || k < 0 || (n > 0 && (!state || !next_state || (k > 0 && (!rewards || !dones)))))
    return HIPENVS_E_ARG;
  if (n == 0) return HIPENVS_OK;
  hipStream_t s = as_stream(stream);
  if (actions)
    hipLaunchKernelGGL(cp::step_k_kernel<true>, dim3(grid_for(n)), dim3(kBlock), 0, s, state, actions, seed, k,
                       next_state, rewards, dones, n);
  else
    hipLaunchKernelGGL(cp::step_k_kernel<false>, dim3(grid_for(n)), dim3(kBlock), 0, s, state, actions, seed, k,
                       next_state, rewards, dones, n);
  return launch_status();
}

extern "C" int hipenvs_sample_actions(int32_t* action, int64_t n, int32_t m, uint32_t seed, hipenvs_stream_t stream) {
  if (n < 0 || m < 1 || m > 256 || (n > 0 && !action)) return HIPENVS_E_ARG;
  if (n == 0) return HIPENVS_OK;
  hipLaunchKernelGGL(cp::sample_actions_kernel, dim3(grid_for(n)), dim3(kBlock), 0, as_stream(stream), action, n,
                     (uint32_t)m, seed);
  return launch_status();
}

extern "C" int hipenvs_cartpole_es_rollout(const float* state, const float* theta, int64_t p, int32_t hidden,
                                           int32_t horizon, float* fitness, hipenvs_stream_t stream) {
  if (p < 0 || horizon < 0 || (p > 0 && (!state || !theta || !fitness))) return HIPENVS_E_ARG;
  if (p == 0) return HIPENVS_OK;
  hipStream_t s = as_stream(stream);
  switch (hidden) {
    case 4: return cp::launch_rollout<4>(state, theta, p, horizon, fitness, s);
    case 8: return cp::launch_rollout<8>(state, theta, p, horizon, fitness, s);
    case 16: return cp::launch_rollout<16>(state, theta, p, horizon, fitness, s);
    case 32: return cp::launch_rollout<32>(state, theta, p, horizon, fitness, s);
    case 64: return cp::launch_rollout<64>(state, theta, p, horizon, fitness, s);
    default: return HIPENVS_E_UNSUPPORTED;
  }
}

extern "C" int hipenvs_cartpole_es_rollout_seeded(const float* state, const float* theta, int64_t p, uint32_t seed,
                                                 double sigma, int32_t hidden, int32_t horizon, float* fitness,
                                                 void* workspace, int64_t workspace_bytes, hipenvs_stream_t stream) {
  if (p < 2 || (p & 1) || p > 0x7fffffffLL || horizon < 0 || !state || !theta || !fitness || !workspace)
    return HIPENVS_E_ARG;
  if (hidden != 4 && hidden != 8 && hidden != 16 && hidden != 32 && hidden != 64) return HIPENVS_E_UNSUPPORTED;
  const int64_t d = 7 * (int64_t)hidden + 2;
  if (workspace_bytes < (int64_t)sizeof(float) * p * d) return HIPENVS_E_ARG;
  float* population = static_cast<float*>(workspace);  // (p, d) rows, written here, read by the rollout
  const int status = launch_perturb(theta, d, p, seed, (float)sigma, kPerturbRows, population, as_stream(stream));
  if (status != HIPENVS_OK) return status;
  return hipenvs_cartpole_es_rollout(state, population, p, hidden, horizon, fitness, stream);
}

extern "C" int hipenvs_cartpole_evaluate(const float* state, const float* theta, int64_t n, int32_t hidden,
                                         int32_t steps, float* fitness, hipenvs_stream_t stream) {
  if (n < 0 || steps < 0 || (n > 0 && (!state || !theta || !fitness))) return HIPENVS_E_ARG;
  if (n == 0) return HIPENVS_OK;
  hipStream_t s = as_stream(stream);
  switch (hidden) {  // every env reads the one policy: member stride 0
    case 4: return cp::launch_rollout<4>(state, theta, 0, n, steps, fitness, s);
    case 8: return cp::launch_rollout<8>(state, theta, 0, n, steps, fitness, s);
    case 16: return cp::launch_rollout<16>(state, theta, 0, n, steps, fitness, s);
    case 32: return cp::launch_rollout<32>(state, theta, 0, n, steps, fitness, s);
    case 64: return cp::launch_rollout<64>(state, theta, 0, n, steps, fitness, s);
    default: return HIPENVS_E_UNSUPPORTED;
  }
}
