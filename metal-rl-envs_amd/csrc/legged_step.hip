// The C-legged body's environment step and reset, and the hopper's (the body at C = 1 with one
// sweep).
#include "legged_body.h"

namespace hipenvs {
namespace lg {

// kHopper (C = 1): the reference's hopper step (hopper_metal.py:84-125): torque
// (a - 1) * TORQUE for any action value, its impulse sum order, and the standing pose
// (0, L, 0, 0) with zero velocities built in (stand is not read).
template <int C, bool kHopper = false>
__global__ __launch_bounds__(kBlock) void step_kernel(const float* __restrict__ state,
                                                      const int32_t* __restrict__ action, uint32_t seed,
                                                      const float* __restrict__ stand, int iters, float assist,
                                                      float assist_damping, float* __restrict__ next,
                                                      float* __restrict__ reward, uint8_t* __restrict__ done,
                                                      int64_t n) {
  constexpr int N = 3 + C;
  const int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (e >= n) return;
  float q[N], v[N], tq[C];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    q[i] = state[i * n + e];
    v[i] = state[(N + i) * n + e];
  }
  // leg k gets ((a / 3^k) % 3 - 1) * TORQUE (legged_np.py:51-54)
  int32_t a = stream_load(action + e);
  if constexpr (kHopper) {
    tq[0] = (float)(a - 1) * TORQUE;
  } else {
#pragma unroll
    for (int k = 0; k < C; ++k) {
      tq[k] = (float)(a % 3 - 1) * TORQUE;
      a /= 3;
    }
  }
#pragma unroll 1
  for (int s = 0; s < SUBSTEPS; ++s) substep_exact<C, kHopper>(q, v, tq, iters, assist, assist_damping);
  const bool d = fallen<C>(q);
  stream_store(d ? 0.0f : v[0] + 1.0f, reward + e);
  stream_store((uint8_t)(d ? 1 : 0), done + e);
  if (d) {  // fresh draws only on fallen lanes; the reference selects (legged_metal.py:148-152)
    const uint32_t h = env_hash(seed, (uint32_t)e);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const float pose = kHopper ? (i == 1 ? 1.0f : 0.0f) : stand[i];  // hopper: y = L = 1
      q[i] = pose + uniform_pm(pcg_hash(h + (uint32_t)i * kRowStride), RESET_BOUND);
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const float pose = kHopper ? 0.0f : stand[N + i];
      v[i] = pose + uniform_pm(pcg_hash(h + (uint32_t)(N + i) * kRowStride), RESET_BOUND);
    }
  }
#pragma unroll
  for (int i = 0; i < N; ++i) next[i * n + e] = q[i];
#pragma unroll
  for (int i = 0; i < N; ++i) next[(N + i) * n + e] = v[i];
}

// The same step with G lanes per env (substep's lane-group form, G = 4 or 16), 64 / G envs to
// a single-wave workgroup. See step_lanes for where it is used and why.
template <int C, int G>
__global__ __launch_bounds__(64) void step_group_kernel(const float* __restrict__ state,
                                                        const int32_t* __restrict__ action, uint32_t seed,
                                                        const float* __restrict__ stand, int iters, float assist,
                                                        float assist_damping, float* __restrict__ next,
                                                        float* __restrict__ reward, uint8_t* __restrict__ done,
                                                        int64_t n) {
  constexpr int N = 3 + C, M = 64 / G;
  __shared__ __align__(16) float xs_all[M * (2 * C + 1) * 8];
  __shared__ __align__(16) float xd_all[M * kBlockFloats<C>];
  const int g = (int)threadIdx.x % G, mloc = (int)threadIdx.x / G;
  float* xs = xs_all + mloc * (2 * C + 1) * 8;
  float* xd = xd_all + mloc * kBlockFloats<C>;
  const int64_t i0 = (int64_t)blockIdx.x * M + mloc;
  const bool live = i0 < n;
  const int64_t e = live ? i0 : n - 1;  // a group past n steps env n - 1, unused: barriers stay uniform
  float q[N], v[N], tq[C];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    q[i] = state[i * n + e];
    v[i] = state[(N + i) * n + e];
  }
  int32_t a = stream_load(action + e);
#pragma unroll
  for (int k = 0; k < C; ++k) {
    tq[k] = (float)(a % 3 - 1) * TORQUE;
    a /= 3;
  }
#pragma unroll 1
  for (int s = 0; s < SUBSTEPS; ++s)
    substep_exact_group<C, G>(q, v, tq, iters, assist, assist_damping, xs, g, live, xd);
  if (!live) return;
  const bool d = fallen<C>(q);
  if (g == 0) {
    stream_store(d ? 0.0f : v[0] + 1.0f, reward + e);
    stream_store((uint8_t)(d ? 1 : 0), done + e);
  }
  const uint32_t h = env_hash(seed, (uint32_t)e);
  // lane g writes rows g, g + G, ...
#pragma unroll
  for (int r0 = 0; r0 < 2 * N; r0 += G) {
    const int r = r0 + g;
    float x = q[r0 < N ? r0 : 0];
#pragma unroll
    for (int i = r0; i < r0 + G && i < 2 * N; ++i) x = (r == i) ? (i < N ? q[i] : v[i - N]) : x;
    if (r < 2 * N) {
      if (d) x = stand[r] + uniform_pm(pcg_hash(h + (uint32_t)r * kRowStride), RESET_BOUND);
      next[r * n + e] = x;
    }
  }
}

template <int C>
__global__ __launch_bounds__(kBlock) void reset_kernel(const float* __restrict__ stand, float* __restrict__ state,
                                                       uint32_t seed, int64_t n) {
  constexpr int N = 3 + C;
  const int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (e >= n) return;
  const uint32_t h = env_hash(seed, (uint32_t)e);
#pragma unroll
  for (int i = 0; i < 2 * N; ++i)
    state[i * n + e] = stand[i] + uniform_pm(pcg_hash(h + (uint32_t)i * kRowStride), RESET_BOUND);
}

// The hopper's reset (hopper_mlx.py:19-20 with the counter RNG of hopper_metal.py:118-120):
// the standing pose (0, L, 0, 0, 0, 0, 0, 0) plus U[+-0.05] on every row.
__global__ __launch_bounds__(kBlock) void hopper_reset_kernel(float* __restrict__ state, uint32_t seed, int64_t n) {
  const int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (e >= n) return;
  const uint32_t h = env_hash(seed, (uint32_t)e);
#pragma unroll
  for (int i = 0; i < 8; ++i)
    state[i * n + e] = (i == 1 ? 1.0f : 0.0f) + uniform_pm(pcg_hash(h + (uint32_t)i * kRowStride), RESET_BOUND);
}

// Lanes per env. The step is bound by the length of one env's instruction stream while the chip
// is not full, and a lane group shortens that: at one wave per SIMD (16 lanes up to 16 envs per
// CU, 4 up to 64) the chip holds the batch in one go. Past 64 envs per CU one lane per env is at
// most one wave per SIMD where 4 lanes are two or more, and no slower. At C = 2 four lanes
// (4 coupling rows, 4 quotients) are as quick as 16 from the start; one contact has nothing to
// share. Step alone, 8 sweeps, us (HIP graph):
//   C = 4, N =  2,048: 36.6 one lane, 24.9 four, 20.6 sixteen    N = 16,384: 36.8, 27.4, 52.1
//          N =  4,097: 41.1, 25.2, 29.0                          N = 20,000: 36.7, 37.7, 62.0
//   C = 3, N =  4,096: 25.4, 19.0, 17.6   C = 2, N = 4,096: 16.2, 12.6, 13.4
//   C = 2, N = 16,385: 16.2, 18.0, 34.0   C = 1, N = 2,048:  6.0,  7.1, 10.4
template <int C>
inline int step_lanes(int64_t n, int64_t cus) {
  if (C >= 3 && n <= 16 * cus) return 16;
  if (C >= 2 && n <= 64 * cus) return 4;
  return 1;
}

template <int C, int G>
int launch_step_group(const float* state, const int32_t* action, uint32_t seed, const float* stand, int iters,
                      double assist, float* next, float* reward, uint8_t* done, int64_t n, hipStream_t s) {
  hipLaunchKernelGGL((step_group_kernel<C, G>), dim3(grid_for(n, 64 / G)), dim3(64), 0, s, state, action, seed, stand,
                     iters, (float)assist, (float)(0.1 * assist), next, reward, done, n);
  return launch_status();
}

template <int C>
int launch_step(const float* state, const int32_t* action, uint32_t seed, const float* stand, int iters, double assist,
                float* next, float* reward, uint8_t* done, int64_t n, hipStream_t s) {
  if constexpr (C >= 2) {
    int cus = 0;
    const int status = device_cus(&cus);
    if (status != HIPENVS_OK) return status;
    const int lanes = step_lanes<C>(n, cus);
    if constexpr (C >= 3) {
      if (lanes == 16)
        return launch_step_group<C, 16>(state, action, seed, stand, iters, assist, next, reward, done, n, s);
    }
    if (lanes == 4)
      return launch_step_group<C, 4>(state, action, seed, stand, iters, assist, next, reward, done, n, s);
  }
  hipLaunchKernelGGL(step_kernel<C>, dim3(grid_for(n)), dim3(kBlock), 0, s, state, action, seed, stand, iters,
                     (float)assist, (float)(0.1 * assist), next, reward, done, n);
  return launch_status();
}

}  // namespace lg
}  // namespace hipenvs

using namespace hipenvs;

extern "C" int hipenvs_legged_reset(int32_t c, const float* stand, float* state, int64_t n, uint32_t seed,
                                    hipenvs_stream_t stream) {
  if (n < 0 || (n > 0 && (!stand || !state))) return HIPENVS_E_ARG;
  if (n == 0) return HIPENVS_OK;
  hipStream_t s = as_stream(stream);
  const dim3 grid(grid_for(n)), block(kBlock);
  switch (c) {
    case 1: hipLaunchKernelGGL(lg::reset_kernel<1>, grid, block, 0, s, stand, state, seed, n); break;
    case 2: hipLaunchKernelGGL(lg::reset_kernel<2>, grid, block, 0, s, stand, state, seed, n); break;
    case 3: hipLaunchKernelGGL(lg::reset_kernel<3>, grid, block, 0, s, stand, state, seed, n); break;
    case 4: hipLaunchKernelGGL(lg::reset_kernel<4>, grid, block, 0, s, stand, state, seed, n); break;
    default: return HIPENVS_E_UNSUPPORTED;
  }
  return launch_status();
}

extern "C" int hipenvs_legged_step(int32_t c, int32_t iters, double assist, const float* state, const int32_t* action,
                                   uint32_t seed, const float* stand, float* next_state, float* reward, uint8_t* done,
                                   int64_t n, hipenvs_stream_t stream) {
  if (n < 0 || iters < 0 || iters > lg::kMaxIters ||
      (n > 0 && (!state || !action || !stand || !next_state || !reward || !done)))
    return HIPENVS_E_ARG;
  if (n == 0) return HIPENVS_OK;
  hipStream_t s = as_stream(stream);
  switch (c) {
    case 1: return lg::launch_step<1>(state, action, seed, stand, iters, assist, next_state, reward, done, n, s);
    case 2: return lg::launch_step<2>(state, action, seed, stand, iters, assist, next_state, reward, done, n, s);
    case 3: return lg::launch_step<3>(state, action, seed, stand, iters, assist, next_state, reward, done, n, s);
    case 4: return lg::launch_step<4>(state, action, seed, stand, iters, assist, next_state, reward, done, n, s);
    default: return HIPENVS_E_UNSUPPORTED;
  }
}

extern "C" int hipenvs_hopper_reset(float* state, int64_t n, uint32_t seed, hipenvs_stream_t stream) {
  if (n < 0 || (n > 0 && !state)) return HIPENVS_E_ARG;
  if (n == 0) return HIPENVS_OK;
  hipLaunchKernelGGL(lg::hopper_reset_kernel, dim3(grid_for(n)), dim3(kBlock), 0, as_stream(stream), state, seed, n);
  return launch_status();
}

extern "C" int hipenvs_hopper_step(const float* state, const int32_t* action, uint32_t seed, float* next_state,
                                   float* reward, uint8_t* done, int64_t n, hipenvs_stream_t stream) {
  if (n < 0 || (n > 0 && (!state || !action || !next_state || !reward || !done))) return HIPENVS_E_ARG;
  if (n == 0) return HIPENVS_OK;
  // one exact contact solve per substep: the C = 1 body with one sweep, no assist
  hipLaunchKernelGGL((lg::step_kernel<1, true>), dim3(grid_for(n)), dim3(kBlock), 0, as_stream(stream), state, action,
                     seed, nullptr, 1, 0.0f, 0.0f, next_state, reward, done, n);
  return launch_status();
}
