// The C-legged body with hard ground contacts on MI355X: one substep of the physics,
// one lane per environment or a lane group per environment, everything in VGPRs (the group
// forms exchange through LDS and DPP). The env step (legged_step.hip) and the fused rollouts
// (legged.hip) are built on it.
//
// Physics: legged_np.py:57-97 in float32, operation by operation. Per substep:
// foot Jacobians (C sincos), the (3+C)^2 mass matrix, a dense Cholesky reused
// for the free velocity and the 2C columns M^-1 J^T, the C^2 Delassus blocks,
// `iters` sweeps of block projected Gauss-Seidel with the exact single-contact
// solve (hopper_np.py:80-109), semi-implicit Euler. Terms the reference
// multiplies by an exact zero or one are elided where that leaves every value
// unchanged (x * 1 = x, x + (+-0) = x); the order of every remaining operation
// is numpy's.
#pragma once

#include <type_traits>

#include "hipenvs_device.h"

namespace hipenvs {
namespace lg {

constexpr float M_F = 0x1.99999ap-3f;              // float32(0.2)
constexpr float I_T = 0x1.99999ap-4f;              // float32(0.1)
constexpr float GRAVITY = 0x1.39999ap+3f;          // float32(9.8)
constexpr float NEG_M_F = -0x1.99999ap-3f;         // float32(-0.2)
constexpr float H = 0x1.47ae14p-7f;                // float32(0.01)
constexpr float MU = 0x1.666666p-1f;               // float32(0.7)
constexpr float BAUMGARTE_OVER_H = 0x1.4p+4f;      // float32(0.2 / 0.01)
constexpr float FALL_HEIGHT = 0x1.333334p-1f;      // float32(0.6)
constexpr float FALL_ANGLE = 0x1p+0f;              // float32(1.0)
constexpr float RESET_BOUND = 0x1.99999ap-5f;      // float32(0.05)
constexpr float TORQUE = 0x1p+1f;                  // float32(2.0)
constexpr int SUBSTEPS = 4;
constexpr int kMaxIters = 4096;                    // sweeps a caller may ask for

// f(std::integral_constant<int, i>) for i = 0 .. K - 1.
template <int K, int I = 0, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < K) {
    f(std::integral_constant<int, I>{});
    static_for<K, I + 1>(f);
  }
}

// np.maximum(x, 0.0): NaN propagates.
__device__ __forceinline__ float max0(float x) { return (x < 0.0f) ? 0.0f : x; }

// x where x > 0, +0 where it is not, in the integer order of the bits (negative numbers, -0
// and NaNs of negative sign become +0; other NaNs stay). One instruction, which folds a DPP
// broadcast of x when `zero` (0) is in a vector register; a float maximum takes a second one
// to quiet a NaN.
__device__ __forceinline__ float clamp0(float x, int zero = 0) {
  const int b = __float_as_int(x);
  return __int_as_float(b > zero ? b : zero);
}

// a where m's bits are set, b where they are not, in the form that becomes one instruction.
__device__ __forceinline__ float bit_select(uint32_t m, float a, float b) {
  const uint32_t y = __float_as_uint(b);
  return __uint_as_float(((__float_as_uint(a) ^ y) & m) ^ y);
}

// Exact impulse of one contact given its Delassus block and relative velocity
// (hopper_np.py:80-109), float32 throughout.
// The per-substep constants of one contact's diagonal Delassus block: the 2x2 determinant
// and the two cone-edge denominators with their float64 reciprocals, formed once per
// substep instead of once per sweep (the values are the same float32 numbers either way).
struct ContactBlock {
  float Att, Atn, Ann, det, den_p, den_m;
  double rdet, rden_p, rden_m;
};

__device__ __forceinline__ ContactBlock contact_block(float Att, float Atn, float Ann) {
  ContactBlock b;
  b.Att = Att;
  b.Atn = Atn;
  b.Ann = Ann;
  b.det = Att * Ann - Atn * Atn;
  b.den_p = Ann + MU * Atn;
  b.den_m = Ann - MU * Atn;
  b.rdet = recip(b.det);
  b.rden_p = recip(b.den_p);
  b.rden_m = recip(b.den_m);
  return b;
}

// What a contact's depth fixes for all sweeps of a substep, for the lane groups: target =
// 20 max(depth, 0), and `closed`, which target - wn must exceed for the contact to push: 0, or
// +inf off the ground. That is touching && wn < target as one compare of the difference, whose
// sign is exact (no difference of two unequal floats rounds to 0). Shut, a contact may not stick
// (the sweep makes its cone NaN wide) and its edges are 0 by themselves: their numerator is 0.
struct ContactGate {
  float target, closed;
};

// The contact's gate. A cone edge has no impulse when its denominator is not positive or the
// foot is off the ground: its reciprocal becomes -2^-300, so that the quotient of its numerator
// (target - wn or 0) is -0 or -inf, or all is NaN, and the sweep's clamp at 0 needs no mask.
__device__ __forceinline__ ContactGate contact_gate(ContactBlock& b, float depth) {
  const bool touching = depth >= 0.0f;
  b.rden_p = (b.den_p > 0.0f && touching) ? b.rden_p : -0x1p-300;
  b.rden_m = (b.den_m > 0.0f && touching) ? b.rden_m : -0x1p-300;
  return ContactGate{BAUMGARTE_OVER_H * max0(depth), touching ? 0.0f : __builtin_inff()};
}

template <class Div>
__device__ __forceinline__ void contact_impulse(const ContactBlock& b, float wt, float wn, float depth,
                                                float& lt_out, float& ln_out, Div& div) {
  const float Att = b.Att, Atn = b.Atn, Ann = b.Ann;
  const bool touching = depth >= 0.0f;
  const float target = BAUMGARTE_OVER_H * max0(depth);
  const float tw = target - wn;
  const float ln_stick = div(Att * tw + Atn * wt, b.det, b.rdet);
  const float lt_stick = div((-Ann) * wt - Atn * tw, b.det, b.rdet);
  const bool sticks = fabsf(lt_stick) <= MU * ln_stick;
  // both cone quotients are formed whatever the signs of their denominators and selected
  // after (no branch); a subnormal mark from an unused one only costs an exact redo
  const float q_p = div(tw, b.den_p, b.rden_p);
  const float q_m = div(tw, b.den_m, b.rden_m);
  const float ln_p = (b.den_p > 0.0f) ? max0(q_p) : 0.0f;
  const float ln_m = (b.den_m > 0.0f) ? max0(q_m) : 0.0f;
  const float slip_p = wt + (Att * MU + Atn) * ln_p;
  const float s = (slip_p <= 0.0f) ? 1.0f : -1.0f;
  const float ln_slide = (slip_p <= 0.0f) ? ln_p : ln_m;
  const float lt_slide = (MU * s) * ln_slide;
  const float ln = sticks ? ln_stick : ln_slide;
  const float lt = sticks ? lt_stick : lt_slide;
  const bool active = touching && (ln > 0.0f) && (wn < target);
  lt_out = active ? lt : 0.0f;
  ln_out = active ? ln : 0.0f;
}

// Solve L L^T x = b in place (pendulum_np.py:95-107): forward then backward substitution.
// rL[i] = recip(L[i][i]): the 2N divisions of a solve share the N diagonal reciprocals.
template <int N, class Div>
__device__ __forceinline__ void chol_solve(const float (&L)[N][N], const double (&rL)[N], float (&b)[N], Div& div) {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    float s = b[i];
#pragma unroll
    for (int p = 0; p < i; ++p) s = s - L[i][p] * b[p];
    b[i] = div(s, L[i][i], rL[i]);
  }
#pragma unroll
  for (int i = N - 1; i >= 0; --i) {
    float s = b[i];
#pragma unroll
    for (int p = i + 1; p < N; ++p) s = s - L[p][i] * b[p];
    b[i] = div(s, L[i][i], rL[i]);
  }
}

// sa[k], ca[k] = lane k * kStride's sn, cs, for k < K, on every lane of the G-lane group.
template <int G, int K, int kStride>
__device__ __forceinline__ void row_trig(float sn, float cs, float* sa, float* ca) {
  if constexpr (K > 0) {
    row_trig<G, K - 1, kStride>(sn, cs, sa, ca);
    sa[K - 1] = lane_bcast<G, (K - 1) * kStride>(sn);
    ca[K - 1] = lane_bcast<G, (K - 1) * kStride>(cs);
  }
}

// out[i] = lane i's x, for i < K, on every lane of the G-lane group.
template <int G, int K>
__device__ __forceinline__ void row_gather(float x, float* out) {
  if constexpr (K > 0) {
    row_gather<G, K - 1>(x, out);
    out[K - 1] = lane_bcast<G, K - 1>(x);
  }
}

// LDS floats per member for the group substep's Delassus and contact blocks (xd)
template <int C>
constexpr int kBlockFloats = 4 * C * C + 12 * C;

// One semi-implicit Euler substep with block PGS contacts, in place (legged_np.py:57-97).
// kGroup = 0: one lane computes the whole substep. kGroup = G (4, 8 or 16): the G lanes
// g = 0..G-1 of a member's group (a DPP quad, a 16-lane DPP row or half of one) all hold the
// member's state and compute everything identically, except that the lanes share by DPP
// broadcast the feet's sines and cosines, one foot a lane, split the 2C + 1 triangular solves
// (the forces and the Jacobian's columns), the C^2 Delassus blocks, the Gauss-Seidel sweeps and
// the velocity update between them (below), and exchange the solves through the group's LDS
// rows xs ((2C + 1) x 8 floats: forces, tangent columns, normal columns) and the blocks through
// xd. Every value is computed by the same expression as in the one-lane form, so the results
// are the same bits. Callers keep the group's lanes in one single-wave workgroup, so the
// barriers order its LDS traffic.
// kHopperSum (C = 1 only) adds the impulse terms as the reference's hopper does,
// (v_free + M^-1 J_t^T lt) + M^-1 J_n^T ln (hopper_np.py:76), instead of the legged body's
// v_free + (M^-1 J_t^T lt + M^-1 J_n^T ln) (legged_np.py:95); otherwise the hopper is this
// body at C = 1 with one sweep.
// kStage (one-lane form only) parks the M^-1 J^T columns in LDS during the Gauss-Seidel
// sweeps, at xs[e * 64] for element e (xs points at the lane's own column of a 64-lane
// block), which frees 2C(3 + C) registers there; they are read back for the velocity update.
template <int C, class Div, int kGroup = 0, bool kHopperSum = false, bool kStage = false>
__device__ __forceinline__ void substep(float (&q)[3 + C], float (&v)[3 + C], const float (&tq)[C], int iters,
                                        float assist, float assist_damping, Div& div, float* xs = nullptr,
                                        int g = 0, float* xd = nullptr) {
  constexpr int N = 3 + C;
  float ca[C], sa[C], dx[C], dy[C], depth[C], r2[C];
  // kRows: every lane has a coupling row of its own, row g % 2C (contact g % 2C / 2, tangential or
  // normal as g is even or odd), and evaluates its contact's sin and cos: its right-hand side,
  // its Delassus blocks, its gate and its free velocity then need no selection among the feet:
  // 885 -> 790 instructions a substep beside the sweeps (16 lanes, C = 4), quadruped step at
  // N = 2,048 21.1 -> 20.0 us.
  constexpr bool kRows = kGroup >= 2 * C && 2 * (kGroup / (2 * C)) >= C;
  const int krow = kRows ? g % (2 * C) : 0, kown = krow / 2;
  const bool nown = krow % 2 != 0;
  float sn = 0.0f, cs = 0.0f;  // of the lane's own foot
  if constexpr (kGroup >= 4 && kGroup >= C) {
    // shared by DPP broadcast within the group, from lane 2k or (not kRows) lane k
    static_assert(C <= kGroup, "one lane per foot");
    float a = q[2] + q[3];
#pragma unroll
    for (int k = 1; k < C; ++k) a = ((kRows ? kown : g) == k) ? q[2] + q[3 + k] : a;
    det_sincos(a, &sn, &cs);
    row_trig<kGroup, C, kRows ? 2 : 1>(sn, cs, sa, ca);
  } else {
#pragma unroll
    for (int k = 0; k < C; ++k) det_sincos(q[2] + q[3 + k], &sa[k], &ca[k]);
  }
#pragma unroll
  for (int k = 0; k < C; ++k) {
    const float ad = v[2] + v[3 + k];
    dx[k] = ((-sa[k]) * ad) * ad;
    dy[k] = (ca[k] * ad) * ad;
    depth[k] = -(q[1] - ca[k]);
    r2[k] = ca[k] * ca[k] + sa[k] * sa[k];
  }
  // sums over the feet in the reference's order
  float s_ca = ca[0], s_sa = sa[0], s_r2 = r2[0], s_dx = dx[0], s_dy = dy[0], s_f2 = ca[0] * dx[0] + sa[0] * dy[0];
#pragma unroll
  for (int k = 1; k < C; ++k) {
    s_ca = s_ca + ca[k];
    s_sa = s_sa + sa[k];
    s_r2 = s_r2 + r2[k];
    s_dx = s_dx + dx[k];
    s_dy = s_dy + dy[k];
    s_f2 = s_f2 + (ca[k] * dx[k] + sa[k] * dy[k]);
  }
  // mass matrix, lower triangle (M_T = 1: base 1 + M_F * C on x and y)
  float L[N][N];
  const float mxy = 1.0f + M_F * (float)C;
  L[0][0] = mxy;
  L[1][0] = M_F * 0.0f;
  L[1][1] = mxy;
  L[2][0] = M_F * s_ca;
  L[2][1] = M_F * s_sa;
  L[2][2] = I_T + M_F * s_r2;
#pragma unroll
  for (int j = 0; j < C; ++j) {
    L[3 + j][0] = M_F * ca[j];
    L[3 + j][1] = M_F * sa[j];
    L[3 + j][2] = M_F * r2[j];
#pragma unroll
    for (int i = 0; i < j; ++i) L[3 + j][3 + i] = M_F * 0.0f;
    L[3 + j][3 + j] = M_F * r2[j];
  }
  // generalised forces: bias, gravity, leg torques, torso assist
  float f[N];
  f[0] = NEG_M_F * s_dx;
  f[1] = NEG_M_F * s_dy - GRAVITY * (M_F * (float)C + 1.0f);
  f[2] = NEG_M_F * s_f2 - GRAVITY * (M_F * s_sa);
#pragma unroll
  for (int j = 0; j < C; ++j) {
    f[3 + j] = NEG_M_F * (ca[j] * dx[j] + sa[j] * dy[j]) - GRAVITY * (M_F * sa[j]);
    f[3 + j] = f[3 + j] + tq[j];
  }
  f[2] = (f[2] - assist * q[2]) - assist_damping * v[2];
  // Cholesky in place (pendulum_np.py:88-94), keeping each pivot's float64 reciprocal
  double rL[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
#pragma unroll
    for (int j = 0; j <= i; ++j) {
      float s = L[i][j];
#pragma unroll
      for (int p = 0; p < j; ++p) s = s - L[i][p] * L[j][p];
      if (i == j) {
        L[i][i] = div.root(s, &rL[i]);
      } else {
        L[i][j] = div(s, L[j][j], rL[j]);
      }
    }
  }
  // M^-1 f and the M^-1 J^T columns
  float MiJt[C][N], MiJn[C][N];
  if constexpr (kGroup == 0) {
    chol_solve<N>(L, rL, f, div);
#pragma unroll
    for (int k = 0; k < C; ++k) {
#pragma unroll
      for (int i = 0; i < N; ++i) {
        MiJt[k][i] = (i == 0) ? 1.0f : (i == 2 || i == 3 + k) ? ca[k] : 0.0f;
        MiJn[k][i] = (i == 1) ? 1.0f : (i == 2 || i == 3 + k) ? sa[k] : 0.0f;
      }
      chol_solve<N>(L, rL, MiJt[k], div);
      chol_solve<N>(L, rL, MiJn[k], div);
    }
  } else {
    constexpr int kRow = 8;  // LDS floats per right-hand side
    constexpr int kRhs = 2 * C + 1, kRounds = (kRhs + kGroup - 1) / kGroup;
    float b[kRounds][N];
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
      if constexpr (kRows) {
        // the lane's own row's column in the first round; the forces on the lanes past 2C, or
        // on all of them in a second round when there are none
        const bool force = g + r * kGroup >= 2 * C;
        const float c = nown ? sn : cs;
#pragma unroll
        for (int i = 0; i < N; ++i) {
          const float j = (i == 0) ? (nown ? 0.0f : 1.0f)
                          : (i == 1) ? (nown ? 1.0f : 0.0f)
                          : (i == 2) ? c : (kown == i - 3) ? c : 0.0f;
          b[r][i] = force ? f[i] : j;
        }
      } else {
        // lane g solves right-hand sides g, g + kGroup, ...; past 2C it solves the forces again, unused
        const int rhs = g + r * kGroup < kRhs ? g + r * kGroup : 0;
        const bool normal = rhs > C;
        const int k = normal ? rhs - 1 - C : rhs - 1;
        float ck = ca[0], sk = sa[0];
#pragma unroll
        for (int kk = 1; kk < C; ++kk) {
          ck = (k == kk) ? ca[kk] : ck;
          sk = (k == kk) ? sa[kk] : sk;
        }
#pragma unroll
        for (int i = 0; i < N; ++i) {
          const bool on = (i == 2 || i == 3 + k);
          const float jt = (i == 0) ? 1.0f : on ? ck : 0.0f;
          const float jn = (i == 1) ? 1.0f : on ? sk : 0.0f;
          b[r][i] = (rhs == 0) ? f[i] : normal ? jn : jt;
        }
      }
      chol_solve<N>(L, rL, b[r], div);
    }
    __syncthreads();  // the rows' previous readers are done
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
      const int h = g + r * kGroup;
      if (h < kRhs) {
        // rows of xs: the forces, the tangent columns, the normal columns
        const int row = !kRows ? h : h == 2 * C ? 0 : 1 + h / 2 + (h % 2) * C;
#pragma unroll
        for (int i = 0; i < N; ++i) xs[row * kRow + i] = b[r][i];
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; ++i) f[i] = xs[i];
    // the M^-1 J^T columns stay in xs until the velocity update reads them
  }
  float vf[N];
#pragma unroll
  for (int i = 0; i < N; ++i) vf[i] = v[i] + H * f[i];
  // Delassus blocks A[k][l] = (Jt_k.MiJt_l, Jt_k.MiJn_l, Jn_k.MiJt_l, Jn_k.MiJn_l) and free velocities
  float Att[C][C], Atn[C][C], Ant[C][C], Ann[C][C], w0t[C], w0n[C];
  if constexpr (kGroup > 0) {
    // lane g < C^2 forms block (g / C, g % C) from the solved rows in xs, and a lane of a
    // diagonal block also forms its contact's ContactBlock; the group reads the C^2 blocks
    // (4 floats each) and the C contact blocks (12 floats each) back from xd
    constexpr int kRow = 8;
    constexpr int kBlocks = C * C, kRounds = kRows ? 1 : (kBlocks + kGroup - 1) / kGroup;
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
      int kb, lb;
      bool mine;
      float ck, sk;
      if constexpr (kRows) {  // row kown's blocks, 2 to each set of 2C lanes
        kb = kown;
        lb = 2 * (g / (2 * C)) + g % 2;
        mine = lb < C;
        lb = mine ? lb : 0;
        ck = cs;
        sk = sn;
      } else {
        const int gr = g + r * kGroup;
        mine = gr < kBlocks;
        const int gb = mine ? gr : 0;  // lanes past C^2 form block 0 again, unused
        kb = gb / C;
        lb = gb % C;
        ck = ca[0];
        sk = sa[0];
#pragma unroll
        for (int kk = 1; kk < C; ++kk) {
          ck = (kb == kk) ? ca[kk] : ck;
          sk = (kb == kk) ? sa[kk] : sk;
        }
      }
      const float* rt = xs + (1 + lb) * kRow;
      const float* rn = xs + (1 + C + lb) * kRow;
      const float t2 = rt[2], t3 = rt[3 + kb], n2 = rn[2], n3 = rn[3 + kb];
      const float4 blk4 = make_float4((rt[0] + ck * t2) + ck * t3, (rn[0] + ck * n2) + ck * n3,
                                      (rt[1] + sk * t2) + sk * t3, (rn[1] + sk * n2) + sk * n3);
      if (mine) *reinterpret_cast<float4*>(xd + 4 * (kb * C + lb)) = blk4;
      ContactBlock own = contact_block(blk4.x, blk4.y, blk4.w);
      if (mine && kb == lb) {
        const ContactGate gate = contact_gate(own, -(q[1] - ck));
        float* xc = xd + 4 * C * C + 12 * kb;
        *reinterpret_cast<float4*>(xc) = make_float4(own.det, own.den_p, own.den_m, own.Att * MU + own.Atn);
        *reinterpret_cast<double2*>(xc + 4) = make_double2(own.rdet, own.rden_p);
        *reinterpret_cast<double*>(xc + 8) = own.rden_m;
        *reinterpret_cast<float2*>(xc + 10) = make_float2(gate.target, gate.closed);
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < C; ++k) {
#pragma unroll
      for (int l = 0; l < C; ++l) {
        const float4 e = *reinterpret_cast<const float4*>(xd + 4 * (k * C + l));
        Att[k][l] = e.x;
        Atn[k][l] = e.y;
        Ant[k][l] = e.z;
        Ann[k][l] = e.w;
      }
    }
  } else {
#pragma unroll
    for (int k = 0; k < C; ++k) {
#pragma unroll
      for (int l = 0; l < C; ++l) {
        Att[k][l] = (MiJt[l][0] + ca[k] * MiJt[l][2]) + ca[k] * MiJt[l][3 + k];
        Atn[k][l] = (MiJn[l][0] + ca[k] * MiJn[l][2]) + ca[k] * MiJn[l][3 + k];
        Ant[k][l] = (MiJt[l][1] + sa[k] * MiJt[l][2]) + sa[k] * MiJt[l][3 + k];
        Ann[k][l] = (MiJn[l][1] + sa[k] * MiJn[l][2]) + sa[k] * MiJn[l][3 + k];
      }
    }
  }
  float w0own = 0.0f;
  if constexpr (kRows) {
    const float c = nown ? sn : cs;
    float vk = vf[3];
#pragma unroll
    for (int k = 1; k < C; ++k) vk = (kown == k) ? vf[3 + k] : vk;
    w0own = ((nown ? vf[1] : vf[0]) + c * vf[2]) + c * vk;
  } else {
#pragma unroll
    for (int k = 0; k < C; ++k) {
      w0t[k] = (vf[0] + ca[k] * vf[2]) + ca[k] * vf[3 + k];
      w0n[k] = (vf[1] + sa[k] * vf[2]) + sa[k] * vf[3 + k];
    }
  }
  if constexpr (kStage) {
    static_assert(kGroup == 0, "staging is for the one-lane form");
#pragma unroll
    for (int k = 0; k < C; ++k) {
#pragma unroll
      for (int i = 0; i < N; ++i) {
        xs[(k * N + i) * 64] = MiJt[k][i];
        xs[((C + k) * N + i) * 64] = MiJn[k][i];
      }
    }
    asm volatile("" ::: "memory");  // the columns live in LDS until the velocity update
  }
  // block projected Gauss-Seidel, fixed contact order (legged_np.py:88-93). One contact is coupled
  // to no other: every sweep solves it from the same free velocity, so the first is the result.
  const int sweeps = C == 1 ? (iters > 0 ? 1 : 0) : iters;
  float lt[C], ln[C];
  ContactBlock blk[C];
#pragma unroll
  for (int k = 0; k < C; ++k) {
    lt[k] = 0.0f;
    ln[k] = 0.0f;
    if constexpr (kGroup == 0) blk[k] = contact_block(Att[k][k], Atn[k][k], Ann[k][k]);
  }
  if constexpr (kGroup >= 4) {
    // The member's lanes split the sweep's independent work and share the results by DPP
    // broadcast. Lane r % G keeps row r (contact r / 2, tangential or normal as r is even or
    // odd) of the coupling, in kSlots rows a lane when G < 2C: when contact l's impulses are
    // known, every row forms its term of them at once (t[s][l], three instructions a slot
    // instead of three for every pair of contacts), and contact k's sum over the others is two
    // more additions in the reference's order. Lanes 0-3 form the four quotients of the
    // contact solve, ln_stick, lt_stick, (target - wn) / den_p and (target - wn) / den_m
    // (lanes 4 and up repeat lane 0's). Every broadcast value is the expression the one-lane
    // sweep evaluates, so the impulses are the same bits.
    // Each lane reads its own coefficients from the group's LDS blocks at a lane-dependent
    // offset (block (k, l) holds Att, Atn, Ant, Ann; contact k's block holds det, den_p,
    // den_m, the slope of slip and then the three's float64 reciprocals, target and closed), and
    // negates by flipping the sign bit: no per-lane selects, which the compiler had turned into
    // exec-mask branches.
    constexpr int kSlots = (2 * C + kGroup - 1) / kGroup;
    const int sel = (g == 2) ? 1 : (g == 3) ? 2 : 0;       // det, den_p, den_m
    const uint32_t neg = (g == 1) ? 0x80000000u : 0u;
    const int oP = (g == 1) ? 3 : 1, oQ = (g == 1) ? 1 : 0;  // Ann|Atn, Atn|Att
    // What bounds the groups is the length of this serial chain and the instructions beside it,
    // so: no mask on the chain is combined on the scalar unit, which would wait for the vector
    // compare to complete (the gate is one compare before the quotients and works through the
    // cone's width); broadcasts fold into their uses (v_sub, v_mul, v_add, v_max with a DPP
    // operand). 16 lanes, C = 4: about 164 instructions a sweep (145 VALU) where per-pair coupling
    // terms, separate broadcasts and a masked clamp and gate took 203 (182 VALU). Quadruped ES
    // rollout at P = 262,144, H = 64, 1,000 steps, 8 sweeps 30.6 -> 27.1 ms for one population
    // (1.07x to 1.13x, as many members last); generation at
    // P = 1,024, H = 16, every member standing for 500 steps 20.2 -> 17.5 ms (17.05 with a row of the
    // setup per lane too, kRows).
    const bool edge = (g == 2 || g == 3);
    float cA[kSlots][C], cB[kSlots][C], w0x[kSlots], t[kSlots][C];
    float qP[C], qQ[C], qd[C], slipc[C], target[C], closed[C];
    bool qzero[C];
    double qr[C];
#pragma unroll
    for (int s = 0; s < kSlots; ++s) {
      const int row = (s * kGroup + g) % (2 * C);  // lanes past 2C repeat the rows from the first
      const float* xr = xd + 4 * C * (row / 2) + 2 * (row % 2);     // Att, Atn or Ant, Ann of contact row / 2
      w0x[s] = kRows ? w0own : w0t[0];
      if constexpr (!kRows) {
#pragma unroll
        for (int r = 1; r < 2 * C; ++r) w0x[s] = (row == r) ? (r % 2 ? w0n[r / 2] : w0t[r / 2]) : w0x[s];
      }
#pragma unroll
      for (int l = 0; l < C; ++l) {
        cA[s][l] = xr[4 * l];
        cB[s][l] = xr[4 * l + 1];
        t[s][l] = cA[s][l] * lt[l] + cB[s][l] * ln[l];
      }
    }
#pragma unroll
    for (int k = 0; k < C; ++k) {
      // numerators qP * wt + qQ * tw: lane 0 Atn wt + Att tw, which is the reference's
      // Att tw + Atn wt (a rounded sum commutes); lane 1 (-Ann) wt + (-Atn) tw, which is
      // the reference's (-Ann) wt - Atn tw exactly (a - b = a + (-b))
      const float* xb = xd + 4 * (k * C + k);
      qP[k] = __uint_as_float(__float_as_uint(xb[oP]) ^ neg);
      qQ[k] = __uint_as_float(__float_as_uint(xb[oQ]) ^ neg);
      const float* xc = xd + 4 * C * C + 12 * k;
      qd[k] = xc[sel];
      qr[k] = *reinterpret_cast<const double*>(xc + 4 + 2 * sel);
      // lane 2 holds den_p, lane 3 den_m; an edge that has no impulse a negative reciprocal
      // (contact_gate). The sign of a zero edge impulse reaches no result: it is added to wt
      // for a comparison with 0, and it is not positive.
      qzero[k] = !Div::kRecip && edge && qr[k] < 0.0;
      const float2 gate = *reinterpret_cast<const float2*>(xc + 10);
      target[k] = gate.x;
      closed[k] = gate.y;
      slipc[k] = xc[3];
    }
    // in vector registers: 0, so that the clamps fold their broadcasts, and the edge lanes as
    // bits, so that the loop selects by them (on a condition the compiler knows to be
    // invariant it splits the loop into copies for the lanes' roles)
    int zero = 0;
    uint32_t edges = edge ? 0xFFFFFFFFu : 0u;
    asm volatile("" : "+v"(zero), "+v"(edges));
    // lanes that hold the same row or quotient as the first: a second broadcast of the value
    // from there folds into its only use instead of being shared
    constexpr int kTwin = kGroup == 16 && 4 * C <= kGroup ? 2 * C : 0;
    constexpr int kTwinQ = kGroup == 16 ? 4 : 0;
    for (int it = 0; it < sweeps; ++it) {
      static_for<C>([&](auto kc) {
        constexpr int k = decltype(kc)::value, s = 2 * k / kGroup;
        float wx = w0x[s];
        if constexpr (C > 1) {
          float sx = 0.0f;
          bool first = true;
#pragma unroll
          for (int l = 0; l < C; ++l) {
            if (l == k) continue;
            sx = first ? t[s][l] : sx + t[s][l];
            first = false;
          }
          wx = wx + sx;
        }
        constexpr int kT = (2 * k) % kGroup, kN = (2 * k + 1) % kGroup;
        const float wt = lane_bcast<kGroup, kT>(wx);
        const float tw = target[k] - lane_bcast<kGroup, kN>(wx);
        const float mu = (tw > closed[k]) ? MU : __builtin_nanf("");
        float num = bit_select(edges, clamp0(tw), qP[k] * wt + qQ[k] * tw);
        if constexpr (!Div::kRecip) num = qzero[k] ? -1.0f : num;
        const float quo = div(num, (!Div::kRecip && qzero[k]) ? 1.0f : qd[k], qr[k]);
        const float ln_stick = lane_bcast<kGroup, 0>(quo);
        const float lt_stick = lane_bcast<kGroup, 1>(quo);
        const float ln_p = clamp0(lane_bcast<kGroup, 2>(quo), zero);
        const float ln_m = clamp0(lane_bcast<kGroup, 3>(quo), zero);
        const bool sticks = fabsf(lt_stick) <= mu * lane_bcast<kGroup, kTwinQ>(quo);
        const float slip_p = lane_bcast<kGroup, kT + kTwin>(wx) + slipc[k] * ln_p;
        const float sgn = (slip_p <= 0.0f) ? 1.0f : -1.0f;
        const float ln_slide = (slip_p <= 0.0f) ? ln_p : ln_m;
        const float lt_slide = (MU * sgn) * ln_slide;
        const float lnv = sticks ? ln_stick : ln_slide;
        const float ltv = sticks ? lt_stick : lt_slide;
        const bool active = lnv > 0.0f;
        lt[k] = active ? ltv : 0.0f;
        ln[k] = active ? lnv : 0.0f;
        if constexpr (C > 1) {
#pragma unroll
          for (int r = 0; r < kSlots; ++r) t[r][k] = cA[r][k] * lt[k] + cB[r][k] * ln[k];
        }
      });
    }
  } else {
    for (int it = 0; it < sweeps; ++it) {
#pragma unroll
      for (int k = 0; k < C; ++k) {
        float st = 0.0f, sn = 0.0f;
        bool first = true;
#pragma unroll
        for (int l = 0; l < C; ++l) {
          if (l == k) continue;
          const float tt = Att[k][l] * lt[l] + Atn[k][l] * ln[l];
          const float nn = Ant[k][l] * lt[l] + Ann[k][l] * ln[l];
          st = first ? tt : st + tt;
          sn = first ? nn : sn + nn;
          first = false;
        }
        const float wt = (C == 1) ? w0t[k] : w0t[k] + st;
        const float wn = (C == 1) ? w0n[k] : w0n[k] + sn;
        contact_impulse(blk[k], wt, wn, depth[k], lt[k], ln[k], div);
      }
    }
  }
  // v = v_free + sum_k M^-1 J_k^T lambda_k; q += h v
  if constexpr (kStage) {
    asm volatile("" ::: "memory");
#pragma unroll
    for (int k = 0; k < C; ++k) {
#pragma unroll
      for (int i = 0; i < N; ++i) {
        MiJt[k][i] = xs[(k * N + i) * 64];
        MiJn[k][i] = xs[((C + k) * N + i) * 64];
      }
    }
  } else if constexpr (kGroup >= 3 + C && !kHopperSum) {
    // lane i < N forms velocity i (its sum over the contacts in the same order as below,
    // from its own column of the solved rows) and the DPP broadcast gives it to the group
    static_assert(3 + C <= kGroup, "one lane per velocity");
    constexpr int kRow = 8;
    asm volatile("" ::: "memory");  // read here, not held in registers through the sweeps
    const int i = g < N ? g : 0;  // lanes past N form velocity 0 again, unused
    float vfi = vf[0];
#pragma unroll
    for (int r = 1; r < N; ++r) vfi = (i == r) ? vf[r] : vfi;
    float si = xs[(1 + 0) * kRow + i] * lt[0] + xs[(1 + C + 0) * kRow + i] * ln[0];
#pragma unroll
    for (int k = 1; k < C; ++k) si = si + (xs[(1 + k) * kRow + i] * lt[k] + xs[(1 + C + k) * kRow + i] * ln[k]);
    float vn[N];
    row_gather<kGroup, N>(vfi + si, vn);
#pragma unroll
    for (int r = 0; r < N; ++r) {
      v[r] = vn[r];
      q[r] = q[r] + H * vn[r];
    }
    return;
  } else if constexpr (kGroup > 0) {
    constexpr int kRow = 8;
    asm volatile("" ::: "memory");  // read here, not held in registers through the sweeps
#pragma unroll
    for (int k = 0; k < C; ++k) {
#pragma unroll
      for (int i = 0; i < N; ++i) {
        MiJt[k][i] = xs[(1 + k) * kRow + i];
        MiJn[k][i] = xs[(1 + C + k) * kRow + i];
      }
    }
  }
#pragma unroll
  for (int i = 0; i < N; ++i) {
    float vn;
    if constexpr (kHopperSum) {
      static_assert(C == 1, "the hopper has one contact");
      vn = (vf[i] + MiJt[0][i] * lt[0]) + MiJn[0][i] * ln[0];
    } else {
      float s = MiJt[0][i] * lt[0] + MiJn[0][i] * ln[0];
#pragma unroll
      for (int k = 1; k < C; ++k) s = s + (MiJt[k][i] * lt[k] + MiJn[k][i] * ln[k]);
      vn = vf[i] + s;
    }
    v[i] = vn;
    q[i] = q[i] + H * vn;
  }
}

// Whether every foot's angle is finite, so that a mass matrix entry that is not comes from
// det_sincos's range (sqrt_pivot) and not from a NaN or an infinity in the state.
template <int C>
__device__ __forceinline__ bool finite_angles(const float (&q)[3 + C]) {
  bool ok = true;
#pragma unroll
  for (int k = 0; k < C; ++k) ok &= fabsf(q[2] + q[3 + k]) < __builtin_inff();
  return ok;
}

// One substep dividing through the shared float64 reciprocals; a lane on which a quotient
// came out subnormal, or a pivot was 0 or infinite (neither met in practice), redoes the
// substep from its saved state with IEEE division and roots, so the result is always the IEEE
// one. Such a pivot leaves NaN in every velocity from finite angles; once the state itself is
// NaN both forms are.
template <int C, bool kHopperSum = false, bool kStage = false>
__device__ __forceinline__ void substep_exact(float (&q)[3 + C], float (&v)[3 + C], const float (&tq)[C], int iters,
                                              float assist, float assist_damping, float* stage = nullptr) {
  constexpr int N = 3 + C;
  float q0[N], v0[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    q0[i] = q[i];
    v0[i] = v[i];
  }
  DivRecip fast;
  substep<C, DivRecip, 0, kHopperSum, kStage>(q, v, tq, iters, assist, assist_damping, fast, stage);
  const bool nan = v[2] != v[2];
  if (fast.saw_subnormal() | nan) {  // one branch on the ordinary path
    if (fast.saw_subnormal() || finite_angles<C>(q0)) {
#pragma unroll
      for (int i = 0; i < N; ++i) {
        q[i] = q0[i];
        v[i] = v0[i];
      }
      DivIEEE ieee;
      substep<C, DivIEEE, 0, kHopperSum, kStage>(q, v, tq, iters, assist, assist_damping, ieee, stage);
    }
  }
}

// The group form of substep_exact: the fast form, and when any live lane of the wave has to
// redo the substep the whole wave does (identical bits wherever nothing called for it), which
// keeps the group's barriers in uniform control flow.
template <int C, int G>
__device__ __forceinline__ void substep_exact_group(float (&q)[3 + C], float (&v)[3 + C], const float (&tq)[C],
                                                    int iters, float assist, float assist_damping, float* xs, int g,
                                                    bool live, float* xd) {
  constexpr int N = 3 + C;
  float q0[N], v0[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    q0[i] = q[i];
    v0[i] = v[i];
  }
  DivRecip fast;
  substep<C, DivRecip, G>(q, v, tq, iters, assist, assist_damping, fast, xs, g, xd);
  const bool nan = v[2] != v[2];
  if (__any(live & (fast.saw_subnormal() | nan)) &&  // lanes of finished members step on, unused
      __any(live && (fast.saw_subnormal() || (nan && finite_angles<C>(q0))))) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      q[i] = q0[i];
      v[i] = v0[i];
    }
    DivIEEE ieee;
    substep<C, DivIEEE, G>(q, v, tq, iters, assist, assist_damping, ieee, xs, g, xd);
  }
}

template <int C>
__device__ __forceinline__ bool fallen(const float (&q)[3 + C]) {
  return (q[1] < FALL_HEIGHT) || (fabsf(q[2]) > FALL_ANGLE);
}

}  // namespace lg
}  // namespace hipenvs
