// The fused ES rollout of a small body (CartPole, Acrobot): one kernel in which a wave steps
// its members in lane groups of 1, 4 or 16 lanes and hands the survivors on to wider groups
// as members finish.
//
// What bounds it: the vector instructions of a member's step, and, once few members are left,
// that step's latency times the longest episode. Per step of H = 32 CartPole a wave issues
// about 1,530 instructions for 64 one-lane members, 480 for 16 four-lane members and 250 for
// 4 sixteen-lane members: wider groups step sooner (the policy is spread over the lanes) but
// cost more per member (the physics is repeated on every lane). Episodes are heavy-tailed
// (early in training most members fail within a few steps and a few last the whole horizon),
// and a wave lives as long as its longest member. So a wave starts with the fewest lanes per
// member that still fill the chip (the launch rules beside each body), and when at most 16 of
// its one-lane members are left it regroups them 4 lanes each, when at most 4 four-lane
// members are left, 16 lanes each. A member's state and id move through LDS, its weights are
// read again in the new layout. Every value is the same expression in every form, so the
// results are the same bits whatever form a member's steps ran in. Workgroups are one wave
// (two or four waves to a workgroup were no faster).
//
// A wave keeps to its end the registers of the form that needs the most. The one-lane form at
// H = 32 (254) lets two waves share a SIMD, so a population of P = 262,144, 4,096 waves, starts in
// two halves: the second waits for the first half's last members, who step in a form that would
// fit eight waves to a SIMD (60 registers). Early in training such a population takes about 600 us,
// of which the longest episode's 500 steps explain 300 (what P = 4,096 takes to the horizon).
#pragma once

#include "es_noise.h"

namespace hipenvs {
namespace roll {

// Body supplies kIn observations, kOut heads, its 4-float state, and
//   Trig trig<G>(state, g)                      what the observation needs beyond the state
//   void observe(state, trig, obs)              the policy's inputs
//   bool step<G>(state, trig, l, alive, g)      one step under the head values l; whether it ended
//   float score(steps, sign)                    the value written for a finished member
struct State4 {
  float a, b, c, d;
};

// Orders the wave's LDS accesses (which the hardware serves in order within a wave) for the
// compiler: what the lanes wrote before is what they read after. No wave waits for another.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Policy weights of one member (es.unflatten's row: w1 (kIn, H), b1 (H), w2 (H, kOut),
// b2 (kOut)) over its G lanes: lane g holds hidden units g * U .. g * U + U - 1 and sums head
// min(g, kOut - 1). Every unit's and head's sum runs in the one-lane order.
template <class Body, int H, int G>
struct Policy {
  static constexpr int I = Body::kIn, O = Body::kOut, U = H >= G ? H / G : 1;
  static_assert(O <= G, "one head per lane");
  // floats of one member's head terms in LDS; the pad keeps the members' rows on different banks
  static constexpr int kRow = O * H + 4;
  float w1[U][I], b1[U], w2[U][O], b2;

  __device__ __forceinline__ void load(const float* __restrict__ row, int g) {
    const int j0 = g * U < H ? g * U : 0;  // lanes past H hold unit 0, unused
#pragma unroll
    for (int k = 0; k < I; ++k)
#pragma unroll
      for (int u = 0; u < U; ++u) w1[u][k] = row[k * H + j0 + u];
#pragma unroll
    for (int u = 0; u < U; ++u) b1[u] = row[I * H + j0 + u];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int o = 0; o < O; ++o) w2[u][o] = row[(I + 1) * H + (j0 + u) * O + o];
    b2 = row[(I + 1 + O) * H + (g < O ? g : O - 1)];
  }

  // The heads on every lane of the group. Each lane writes its units' terms h_j * w2[j][o] to
  // the member's LDS row (head o's at o * H + j); the head lanes add them in order.
  __device__ __forceinline__ void heads(const float (&obs)[I], float* xp, int g, float (&l)[O]) const {
    float pre[U], h[U];
#pragma unroll
    for (int u = 0; u < U; ++u) pre[u] = obs[0] * w1[u][0];
#pragma unroll
    for (int k = 1; k < I; ++k)
#pragma unroll
      for (int u = 0; u < U; ++u) pre[u] = pre[u] + obs[k] * w1[u][k];
#pragma unroll
    for (int u = 0; u < U; ++u) pre[u] = pre[u] + b1[u];
    det_tanh_all<U>(pre, h);
    if (H >= G || g < H) {
#pragma unroll
      for (int o = 0; o < O; ++o)
#pragma unroll
        for (int u = 0; u < U; ++u) xp[o * H + g * U + u] = h[u] * w2[u][o];
    }
    wave_sync();
    const float* xo = xp + (g < O ? g : O - 1) * H;
    // every read issues before the first sum waits for one (up to 32 at a time)
    float s = b2;
    constexpr int kBatch = H < 32 ? H : 32;
#pragma unroll
    for (int j0 = 0; j0 < H; j0 += kBatch) {
      float v[kBatch];
#pragma unroll
      for (int j = 0; j < kBatch; ++j) v[j] = xo[j0 + j];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < kBatch; ++j) s = s + v[j];
    }
    wave_sync();  // the rows are read before the next step writes them
    l[0] = lane_bcast<G, 0>(s);
    l[1] = lane_bcast<G, 1>(s);
    if constexpr (O > 2) l[2] = lane_bcast<G, 2>(s);
  }
};

template <class Body, int H>
struct Policy<Body, H, 1> {
  static constexpr int I = Body::kIn, O = Body::kOut, D = (I + 1 + O) * H + O;
  float w[D];

  __device__ __forceinline__ void load(const float* __restrict__ row, int) {
#pragma unroll
    for (int d = 0; d < D; ++d) w[d] = row[d];
  }

  __device__ __forceinline__ void heads(const float (&obs)[I], float*, int, float (&l)[O]) const {
#pragma unroll
    for (int o = 0; o < O; ++o) l[o] = w[(I + 1 + O) * H + o];
    // two units' chains at a time: one at a time, two waves on a SIMD took 4,667 us where
    // these take 4,133 (CartPole, trained, P = 262,144, H = 32); four at a time spill at H = 32
    constexpr int kBatch = 2;
#pragma unroll
    for (int j0 = 0; j0 < H; j0 += kBatch) {
      float pre[kBatch], h[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const int j = j0 + u;
        pre[u] = obs[0] * w[j];
#pragma unroll
        for (int k = 1; k < I; ++k) pre[u] = pre[u] + obs[k] * w[k * H + j];
        pre[u] = pre[u] + w[I * H + j];
      }
      det_tanh_all<kBatch>(pre, h);
#pragma unroll
      for (int u = 0; u < kBatch; ++u)
#pragma unroll
        for (int o = 0; o < O; ++o) l[o] = l[o] + h[u] * w[(I + 1) * H + O * (j0 + u) + o];
    }
  }
};

struct Slot {
  State4 s;
  int64_t m;
};

// Steps the wave's members, G lanes each, from step t on while more than `narrow_at` of them
// are live, and writes the score of each as it finishes. A wave's live members are all at
// the same step, so t and the horizon are the wave's. Every lane steps (barriers and
// broadcasts stay uniform); a finished member's results are discarded.
template <class Body, int H, int G>
__device__ __forceinline__ void run(State4& s, int64_t m, int32_t& t, bool& alive, const float* __restrict__ theta,
                                    int64_t member_stride, int32_t horizon, float sign, float* __restrict__ out,
                                    float* lds, int narrow_at) {
  const int g = (int)threadIdx.x % G;
  float* xp = lds;
  if constexpr (G > 1) xp = lds + ((int)threadIdx.x / G) * Policy<Body, H, G>::kRow;
  Policy<Body, H, G> policy;
  policy.load(theta + m * member_stride, g);
  auto trig = Body::template trig<G>(s, g);
  bool live = alive;
  if (__popcll(__builtin_amdgcn_ballot_w64(live)) > narrow_at * G) {
    while (t < horizon) {
      float obs[Body::kIn], l[Body::kOut];
      Body::observe(s, trig, obs);
      policy.heads(obs, xp, g, l);
      const bool ended = Body::template step<G>(s, trig, l, live, g);
      if (__builtin_amdgcn_ballot_w64(live && ended)) {
        if (live && ended && g == 0) out[m] = Body::score(t, sign);
        live = live && !ended;
        if (__popcll(__builtin_amdgcn_ballot_w64(live)) <= narrow_at * G) {
          ++t;
          break;
        }
      }
      ++t;
    }
  }
  if (t >= horizon && live) {
    if (g == 0) out[m] = Body::score(t, sign);
    live = false;
  }
  alive = live;
}

// Regroups the wave's live members (at most 64 / GN of them) from G to GN lanes each.
template <int G, int GN>
__device__ __forceinline__ void narrow(State4& s, int64_t& m, bool& alive, Slot* slots) {
  const int lane = (int)threadIdx.x;
  const unsigned long long live = __builtin_amdgcn_ballot_w64(alive && lane % G == 0);
  if (alive && lane % G == 0) {
    Slot& to = slots[__popcll(live & ((1ull << lane) - 1ull))];
    to.s = s;
    to.m = m;
  }
  wave_sync();
  alive = lane / GN < __popcll(live);
  if (live) {  // lanes past the live members step the first one, unused
    const Slot& from = slots[alive ? lane / GN : 0];
    s = from.s;
    m = from.m;
  }
  wave_sync();
}

template <class Body, int H>
constexpr int kLdsFloats = 16 * Policy<Body, H, 4>::kRow > 4 * Policy<Body, H, 16>::kRow
                               ? 16 * Policy<Body, H, 4>::kRow
                               : 4 * Policy<Body, H, 16>::kRow;

// Whether the form runs populations of any size with more threads than members: at H = 64, 4 lanes
// per member past the 16-lane bound. A grid's x has to stay below 2^32 threads (past that the
// launch reports no error and runs the remainder of the division), which 2^30 members would
// reach: their blocks spread over rows of kMaxBlocksX. (An evaluation of 2^30 envs holds 21 GB.)
template <int H, int G>
constexpr bool kRowedGrid = G == 4 && H > 32;
constexpr int64_t kMaxBlocksX = (1LL << 26) - 1;

// G lanes per member at the start. member_stride D for a population, 0 for one policy shared by
// every env (the greedy evaluation).
template <class Body, int H, int G>
__global__ __launch_bounds__(64, (Body::template kMinWaves<H, G>)) void rollout_kernel(
    const float* __restrict__ state, const float* __restrict__ theta, int64_t member_stride, int64_t p,
    int32_t horizon, float sign, float* __restrict__ out) {
  __shared__ __align__(16) float lds[kLdsFloats<Body, H>];
  __shared__ Slot slots[16];
  constexpr int M = 64 / G;
  int64_t block = blockIdx.x;
  if constexpr (kRowedGrid<H, G>) block += (int64_t)blockIdx.y * gridDim.x;
  const int64_t i = block * M + (int)threadIdx.x / G;
  int64_t m = i < p ? i : p - 1;  // a group past p steps member p - 1, unused
  State4 x{state[m], state[p + m], state[2 * p + m], state[3 * p + m]};
  int32_t t = 0;
  bool alive = i < p;
  if constexpr (G == 1) {
    run<Body, H, 1>(x, m, t, alive, theta, member_stride, horizon, sign, out, lds, 16);
    narrow<1, 4>(x, m, alive, slots);
  }
  if constexpr (G <= 4) {
    run<Body, H, 4>(x, m, t, alive, theta, member_stride, horizon, sign, out, lds, 4);
    narrow<4, 16>(x, m, alive, slots);
  }
  run<Body, H, 16>(x, m, t, alive, theta, member_stride, horizon, sign, out, lds, 0);
}

template <class Body, int H, int G>
int launch(const float* state, const float* theta, int64_t member_stride, int64_t p, int32_t horizon, float sign,
           float* out, hipStream_t s) {
  constexpr int M = 64 / G;
  const int64_t blocks = (p + M - 1) / M;
  const int64_t rows = kRowedGrid<H, G> ? (blocks + kMaxBlocksX - 1) / kMaxBlocksX : 1;
  hipLaunchKernelGGL((rollout_kernel<Body, H, G>), dim3((unsigned)((blocks + rows - 1) / rows), (unsigned)rows),
                     dim3(64), 0, s, state, theta, member_stride, p, horizon, sign, out);
  return launch_status();
}

}  // namespace roll
}  // namespace hipenvs
