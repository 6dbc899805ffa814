// Acrobot on MI355X: the single-step kernel (RK4 at dt 0.2, wrap, clip, masked
// reset) and the fused ES rollout kernel (6-H-3 tanh policy + the same physics
// for the whole horizon in registers), with their C-ABI entry points.
//
// The derivative follows acrobot_np.py:64-84 operation by operation, with the
// Python-scalar products already folded to the float32 constants numpy uses
// (each constant's defining expression is beside it); RK4/wrap/clip follow
// acrobot_np.py:47-61,87-89, termination acrobot_np.py:92-93, reset the
// counter RNG of acrobot_metal.py:78-83. Per env-step the step kernel moves 41
// algorithmic bytes; it is VALU-bound (14 sin/cos, 18 divisions, of which 8
// through a reciprocal estimate).

#include "acrobot_mass.h"
#include "es_rollout.h"

namespace hipenvs {
namespace ac {

constexpr float PHI2_C = 0x1.39999ap+2f;      // float32(1.0 * 0.5 * 9.8)
constexpr float HALF_PI = 0x1.921fb6p+0f;     // float32(pi / 2)
constexpr float PHI1_A = -0x1p-1f;            // float32(-1.0 * 1.0 * 0.5)
constexpr float PHI1_C = 0x1.d66666p+3f;      // float32((1.0 * 0.5 + 1.0 * 1.0) * 9.8)
constexpr float DD2_C = 0x1p-1f;              // float32(1.0 * 1.0 * 0.5)
constexpr float DEN_C = 0x1.4p+0f;            // float32(1.0 * 0.5**2 + 1.0)
constexpr float DT = 0x1.99999ap-3f;          // float32(0.2)
constexpr float DT_2 = 0x1.99999ap-4f;        // float32(0.2 / 2)
constexpr float DT_6 = 0x1.111112p-5f;        // float32(0.2 / 6)
constexpr float TWO_PI = 0x1.921fb6p+2f;      // float32(2 * pi)
constexpr float PI = 0x1.921fb6p+1f;          // float32(pi)
constexpr float MAX_VEL_1 = 0x1.921fb6p+3f;   // float32(4 * pi)
constexpr float MAX_VEL_2 = 0x1.c463acp+4f;   // float32(9 * pi)
constexpr float RESET_BOUND = 0x1.99999ap-4f; // float32(0.1)

using S4 = roll::State4;  // theta1, theta2, dtheta1, dtheta2 (or their derivatives)

// acrobot_np.py:64-84. The numpy expression's multiplications by the Python
// float 1.0 (m2 *, 2 * l1 * lc2 *) are exact and omitted.
// The two quotients of d2 by d1 come from d1's reciprocal estimate (acrobot_mass.h), or with
// kInRange false from IEEE division; `reach` keeps the largest |cos(theta2)| met. The other two
// divide with IEEE division: through a float64 reciprocal, with a wave vote for tiny numerators,
// the step gained nothing (6.37 against 6.22 us at N = 262,144) and the group form lost (874
// against 863 us a rollout). The three sin/cos share one range vote.
template <bool kInRange>
__device__ __forceinline__ S4 dsdt(const S4& s, float torque, float& reach) {
  const float ang[3] = {s.b, (s.a + s.b) - HALF_PI, s.a - HALF_PI};
  float sn[3], cs[3];
  if constexpr (kInRange) {
    det_sincos_small<3>(ang, sn, cs);
  } else {
#pragma unroll
    for (int i = 0; i < 3; ++i) det_sincos(ang[i], &sn[i], &cs[i]);
  }
  const float s2 = sn[0], c2 = cs[0];
  reach = fmaxf(reach, fabsf(c2));
  const float d1 = mass_d1(c2), d2 = mass_d2(c2);
  const float r1 = __builtin_amdgcn_rcpf(d1);
  const float phi2 = PHI2_C * cs[1];
  const float t1 = (PHI1_A * (s.d * s.d)) * s2;
  const float t2 = (s.d * s.c) * s2;
  const float t3 = PHI1_C * cs[2];
  const float phi1 = ((t1 - t2) + t3) + phi2;
  const float num = ((torque + mass_quotient<kInRange>(d2, d1, r1) * phi1) - (DD2_C * (s.c * s.c)) * s2) - phi2;
  const float den = DEN_C - mass_quotient<kInRange>(d2 * d2, d1, r1);
  const float dd2 = num / den;
  const float dd1 = (-((d2 * dd2) + phi1)) / d1;
  return S4{s.c, s.d, dd1, dd2};
}

constexpr double INV_TWO_PI = 1.0 / (double)TWO_PI;  // for div_const(x, .) == x / TWO_PI

__device__ __forceinline__ float wrap(float x) { return x - TWO_PI * floorf(div_const(x + PI, INV_TWO_PI)); }

// The group's physics, with the transcendentals and the two quotients by d1 spread over the
// group's lanes: lanes 0, 1, 2 evaluate one det_sincos each (one instruction stream for the
// three) and every lane of the 16-lane group (one DPP row) receives the results by row
// broadcast. Each value is the single-lane function's on the same argument, so the bits
// are those of dsdt/rk4/terminal.
struct GroupTrig {
  float sin_a, cos_a, sin_b, cos_b, cos_ab;  // theta1, theta2, theta2 + theta1
};

template <int G>
__device__ __forceinline__ GroupTrig group_trig(const S4& s, int g) {
  const float x = (g == 1) ? s.b : (g == 2) ? (s.b + s.a) : s.a;
  float sn, cs;
  det_sincos(x, &sn, &cs);
  return GroupTrig{lane_bcast<G, 0>(sn), lane_bcast<G, 0>(cs), lane_bcast<G, 1>(sn), lane_bcast<G, 1>(cs),
                   lane_bcast<G, 2>(cs)};
}

template <int G, bool kInRange>
__device__ __forceinline__ S4 dsdt_group(const S4& s, float torque, int g, float& reach) {
  const float x = (g == 1) ? ((s.a + s.b) - HALF_PI) : (g == 2) ? (s.a - HALF_PI) : s.b;
  float sn, cs;
  det_sincos(x, &sn, &cs);
  const float s2 = lane_bcast<G, 0>(sn), c2 = lane_bcast<G, 0>(cs);
  reach = fmaxf(reach, fabsf(c2));
  const float d1 = mass_d1(c2), d2 = mass_d2(c2);
  const float phi2 = PHI2_C * lane_bcast<G, 1>(cs);
  const float t1 = (PHI1_A * (s.d * s.d)) * s2;
  const float t2 = (s.d * s.c) * s2;
  const float t3 = PHI1_C * lane_bcast<G, 2>(cs);
  const float phi1 = ((t1 - t2) + t3) + phi2;
  // lane 1: d2^2 / d1, else d2 / d1
  const float q = mass_quotient<kInRange>((g == 1) ? d2 * d2 : d2, d1, __builtin_amdgcn_rcpf(d1));
  const float num = ((torque + lane_bcast<G, 0>(q) * phi1) - (DD2_C * (s.c * s.c)) * s2) - phi2;
  const float den = DEN_C - lane_bcast<G, 1>(q);
  const float dd2 = num / den;
  const float dd1 = (-((d2 * dd2) + phi1)) / d1;
  return S4{s.c, s.d, dd1, dd2};
}

template <int G, bool kInRange>
__device__ __forceinline__ S4 derivative(const S4& s, float torque, int g, float& reach) {
  if constexpr (G == 1)
    return dsdt<kInRange>(s, torque, reach);
  else
    return dsdt_group<G, kInRange>(s, torque, g, reach);
}

// RK4 (acrobot_np.py:47-61) from s, before the wrap and clip. The out-of-range form, which no
// ordinary state takes, is a rolled loop, so that it costs the other neither registers nor the
// instruction cache (unrolled it took 10 registers more: one lane at H = 8 fell from four waves per
// SIMD to three; a choice in each derivative instead, under the sin/cos vote, took the 16-lane
// rollout at P = 4,096 from 806 to 931 us).
template <int G, bool kInRange>
__device__ __forceinline__ S4 rk4_unwrapped(const S4& s, float torque, int g, float& reach) {
  S4 sum{}, x = s;
  if constexpr (kInRange) {
    const S4 k1 = derivative<G, true>(s, torque, g, reach);
    const S4 k2 = derivative<G, true>(
        S4{s.a + DT_2 * k1.a, s.b + DT_2 * k1.b, s.c + DT_2 * k1.c, s.d + DT_2 * k1.d}, torque, g, reach);
    const S4 k3 = derivative<G, true>(
        S4{s.a + DT_2 * k2.a, s.b + DT_2 * k2.b, s.c + DT_2 * k2.c, s.d + DT_2 * k2.d}, torque, g, reach);
    const S4 k4 = derivative<G, true>(
        S4{s.a + DT * k3.a, s.b + DT * k3.b, s.c + DT * k3.c, s.d + DT * k3.d}, torque, g, reach);
    sum = S4{((k1.a + 2.0f * k2.a) + 2.0f * k3.a) + k4.a, ((k1.b + 2.0f * k2.b) + 2.0f * k3.b) + k4.b,
             ((k1.c + 2.0f * k2.c) + 2.0f * k3.c) + k4.c, ((k1.d + 2.0f * k2.d) + 2.0f * k3.d) + k4.d};
  } else {
#pragma unroll 1
    for (int i = 0; i < 4; ++i) {
      const S4 k = derivative<G, false>(x, torque, g, reach);
      const float w = (i == 1 || i == 2) ? 2.0f : 1.0f, h = (i == 2) ? DT : DT_2;
      sum = S4{i ? sum.a + w * k.a : k.a, i ? sum.b + w * k.b : k.b, i ? sum.c + w * k.c : k.c,
               i ? sum.d + w * k.d : k.d};
      x = S4{s.a + h * k.a, s.b + h * k.b, s.c + h * k.c, s.d + h * k.d};
    }
  }
  return S4{s.a + DT_6 * sum.a, s.b + DT_6 * sum.b, s.c + DT_6 * sum.c, s.d + DT_6 * sum.d};
}

// RK4 + wrap + clip in place (acrobot_np.py:47-61) on G lanes. When a cosine on any lane left the
// range that the short quotients are exact over (angles past about 2^50, see acrobot_mass.h), the
// wave evaluates again with IEEE division: the same bits for the others.
template <int G>
__device__ __forceinline__ void rk4(S4& s, float torque, int g = 0) {
  float reach = 0.0f;
  S4 x = rk4_unwrapped<G, true>(s, torque, g, reach);
  if (__builtin_expect(!wave_all(!(reach > kMassRange)), 0)) x = rk4_unwrapped<G, false>(s, torque, g, reach);
  s.a = wrap(x.a);
  s.b = wrap(x.b);
  s.c = clip(x.c, -MAX_VEL_1, MAX_VEL_1);
  s.d = clip(x.d, -MAX_VEL_2, MAX_VEL_2);
}

// acrobot_np.py:92-93: -cos(th1) - cos(th2 + th1) > 1.
__device__ __forceinline__ bool terminal(const S4& s) {
  const float ang[2] = {s.a, s.b + s.a};
  float sn[2], cs[2];
  det_sincos_small<2>(ang, sn, cs);
  return (-cs[0]) - cs[1] > 1.0f;
}

__global__ __launch_bounds__(kBlock) void reset_kernel(float* __restrict__ state, uint32_t seed, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const uint32_t h = env_hash(seed, (uint32_t)i);
  state[i] = uniform_pm(pcg_hash(h), RESET_BOUND);
  state[n + i] = uniform_pm(pcg_hash(h + kRowOff1), RESET_BOUND);
  state[2 * n + i] = uniform_pm(pcg_hash(h + kRowOff2), RESET_BOUND);
  state[3 * n + i] = uniform_pm(pcg_hash(h + kRowOff3), RESET_BOUND);
}

__global__ __launch_bounds__(kBlock) void step_kernel(const float* __restrict__ state, const int32_t* __restrict__ action,
                                                      uint32_t seed, float* __restrict__ next, float* __restrict__ reward,
                                                      uint8_t* __restrict__ done, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  S4 s{state[i], state[n + i], state[2 * n + i], state[3 * n + i]};
  const float torque = (float)(stream_load(action + i) - 1);
  rk4<1>(s, torque);
  const bool d = terminal(s);
  if (d) {  // fresh draws only on terminated lanes; the reference selects (acrobot_metal.py:76-80)
    const uint32_t h = env_hash(seed, (uint32_t)i);
    s.a = uniform_pm(pcg_hash(h), RESET_BOUND);
    s.b = uniform_pm(pcg_hash(h + kRowOff1), RESET_BOUND);
    s.c = uniform_pm(pcg_hash(h + kRowOff2), RESET_BOUND);
    s.d = uniform_pm(pcg_hash(h + kRowOff3), RESET_BOUND);
  }
  next[i] = s.a;
  next[n + i] = s.b;
  next[2 * n + i] = s.c;
  next[3 * n + i] = s.d;
  stream_store(d ? 0.0f : -1.0f, reward + i);
  stream_store((uint8_t)(d ? 1 : 0), done + i);
}

// The fused ES rollout's body (es_rollout.h): Gym's observation, the 6-H-3 tanh policy with
// first-index argmax over three torques, RK4 physics, stop at the first termination
// (acrobot_rollout_metal.py:21-58). A population's score is the steps survived (sign 1), the
// greedy evaluation's minus the steps (sign -1).
struct RolloutBody {
  static constexpr int kIn = 6, kOut = 3;
  template <int H, int G>
  static constexpr int kMinWaves = 1;
  using Trig = GroupTrig;  // the observation's trig; after each step also the termination's
  template <int G>
  __device__ static __forceinline__ Trig trig(const S4& s, int g) {
    if constexpr (G == 1) {
      Trig t;
      det_sincos(s.a, &t.sin_a, &t.cos_a);
      det_sincos(s.b, &t.sin_b, &t.cos_b);
      t.cos_ab = det_cos(s.b + s.a);
      return t;
    } else {
      return group_trig<G>(s, g);
    }
  }
  __device__ static __forceinline__ void observe(const S4& s, const Trig& t, float (&obs)[6]) {
    obs[0] = t.cos_a;
    obs[1] = t.sin_a;
    obs[2] = t.cos_b;
    obs[3] = t.sin_b;
    obs[4] = s.c;
    obs[5] = s.d;
  }
  template <int G>
  __device__ static __forceinline__ bool step(S4& s, Trig& t, const float (&l)[3], bool, int g) {
    float torque = -1.0f, best = l[0];
    if (l[1] > best) { torque = 0.0f; best = l[1]; }
    if (l[2] > best) { torque = 1.0f; }
    rk4<G>(s, torque, g);
    t = trig<G>(s, g);
    return (-t.cos_a) - t.cos_ab > 1.0f;  // terminal(s)
  }
  // steps as a float32 count that stops at 2^24, where adding one no longer changes it; + 0: a
  // score of -0 reads +0
  __device__ static __forceinline__ float score(int32_t t, float sign) {
    return sign * (float)(t < 0x1000000 ? t : 0x1000000) + 0.0f;
  }
};

// Lanes per member at the start, by members per CU (500 steps, most members run them all; P
// on 256 CUs, us; 16 / 4 / 1 lanes):
//   H = 32: P = 4,096 826 / 1,074 / 2,455; 8,192 1,262 / 1,128 / 2,464; 32,768 4,594 / 1,973 /
//           2,507; 65,536 8,044 / 2,960 / 2,503; 262,144 29,660 / 10,715 / 9,938
//   H = 8:  P = 4,096 795 / 778 / 1,305; 32,768 3,619 / 1,141 / 1,330; 65,536 6,849 / 2,148 / 1,317
//   H = 64: P = 32,768 5,694 / 2,319, one lane 5,108; 262,144 16,475, one lane 26,696
constexpr int kGroup16PerCu = 16, kGroup4PerCu = 128;

template <int H>
int launch_rollout(const float* state, const float* theta, int64_t member_stride, int64_t p, int32_t horizon,
                   float sign, float* out, hipStream_t s) {
  int cus = 0;
  const int status = device_cus(&cus);
  if (status != HIPENVS_OK) return status;
  if (p <= (int64_t)kGroup16PerCu * cus)
    return roll::launch<RolloutBody, H, 16>(state, theta, member_stride, p, horizon, sign, out, s);
  if (H > 32 || p <= (int64_t)kGroup4PerCu * cus)
    return roll::launch<RolloutBody, H, 4>(state, theta, member_stride, p, horizon, sign, out, s);
  return roll::launch<RolloutBody, H, (H > 32 ? 4 : 1)>(state, theta, member_stride, p, horizon, sign, out, s);
}

template <int H>
int launch_rollout(const float* state, const float* theta, int64_t p, int32_t horizon, float* out, hipStream_t s) {
  return launch_rollout<H>(state, theta, (int64_t)(10 * H + 3), p, horizon, 1.0f, out, s);
}

}  // namespace ac
}  // namespace hipenvs

using namespace hipenvs;

extern "C" int hipenvs_acrobot_reset(float* state, int64_t n, uint32_t seed, hipenvs_stream_t stream) {
  if (n < 0 || (n > 0 && !state)) return HIPENVS_E_ARG;
  if (n == 0) return HIPENVS_OK;
  hipLaunchKernelGGL(ac::reset_kernel, dim3(grid_for(n)), dim3(kBlock), 0, as_stream(stream), state, seed, n);
  return launch_status();
}

extern "C" int hipenvs_acrobot_step(const float* state, const int32_t* action, uint32_t seed, float* next_state,
                                    float* reward, uint8_t* done, int64_t n, hipenvs_stream_t stream) {
  if (n < 0 || (n > 0 && (!state || !action || !next_state || !reward || !done))) return HIPENVS_E_ARG;
  if (n == 0) return HIPENVS_OK;
  hipLaunchKernelGGL(ac::step_kernel, dim3(grid_for(n)), dim3(kBlock), 0, as_stream(stream), state, action, seed,
                     next_state, reward, done, n);
  return launch_status();
}

extern "C" int hipenvs_acrobot_es_rollout(const float* state, const float* theta, int64_t p, int32_t hidden,
                                          int32_t horizon, float* steps, hipenvs_stream_t stream) {
  if (p < 0 || horizon < 0 || (p > 0 && (!state || !theta || !steps))) return HIPENVS_E_ARG;
  if (p == 0) return HIPENVS_OK;
  hipStream_t s = as_stream(stream);
  switch (hidden) {
    case 4: return ac::launch_rollout<4>(state, theta, p, horizon, steps, s);
    case 8: return ac::launch_rollout<8>(state, theta, p, horizon, steps, s);
    case 16: return ac::launch_rollout<16>(state, theta, p, horizon, steps, s);
    case 32: return ac::launch_rollout<32>(state, theta, p, horizon, steps, s);
    case 64: return ac::launch_rollout<64>(state, theta, p, horizon, steps, s);
    default: return HIPENVS_E_UNSUPPORTED;
  }
}

extern "C" int hipenvs_acrobot_es_rollout_seeded(const float* state, const float* theta, int64_t p, uint32_t seed,
                                                 double sigma, int32_t hidden, int32_t horizon, float* steps,
                                                 void* workspace, int64_t workspace_bytes, hipenvs_stream_t stream) {
  if (p < 2 || (p & 1) || p > 0x7fffffffLL || horizon < 0 || !state || !theta || !steps || !workspace)
    return HIPENVS_E_ARG;
  if (hidden != 4 && hidden != 8 && hidden != 16 && hidden != 32 && hidden != 64) return HIPENVS_E_UNSUPPORTED;
  const int64_t d = 10 * (int64_t)hidden + 3;
  if (workspace_bytes < (int64_t)sizeof(float) * p * d) return HIPENVS_E_ARG;
  float* population = static_cast<float*>(workspace);  // (p, d) rows, written here, read by the rollout
  const int status = launch_perturb(theta, d, p, seed, (float)sigma, kPerturbRows, population, as_stream(stream));
  if (status != HIPENVS_OK) return status;
  return hipenvs_acrobot_es_rollout(state, population, p, hidden, horizon, steps, stream);
}

extern "C" int hipenvs_acrobot_evaluate(const float* state, const float* theta, int64_t n, int32_t hidden,
                                        int32_t steps, float* fitness, hipenvs_stream_t stream) {
  if (n < 0 || steps < 0 || (n > 0 && (!state || !theta || !fitness))) return HIPENVS_E_ARG;
  if (n == 0) return HIPENVS_OK;
  hipStream_t s = as_stream(stream);
  switch (hidden) {  // every env reads the one policy: member stride 0; score = -steps
    case 4: return ac::launch_rollout<4>(state, theta, 0, n, steps, -1.0f, fitness, s);
    case 8: return ac::launch_rollout<8>(state, theta, 0, n, steps, -1.0f, fitness, s);
    case 16: return ac::launch_rollout<16>(state, theta, 0, n, steps, -1.0f, fitness, s);
    case 32: return ac::launch_rollout<32>(state, theta, 0, n, steps, -1.0f, fitness, s);
    case 64: return ac::launch_rollout<64>(state, theta, 0, n, steps, -1.0f, fitness, s);
    default: return HIPENVS_E_UNSUPPORTED;
  }
}
