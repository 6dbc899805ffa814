"""The calls a user of hipenvs makes, as measurable cases: what is called, on which inputs,
what the path cannot do without, and its result in 64 bits.

Four kinds of call carry the framework's main path:

* one environment step of a batch (``step``): a learner's inner loop, from a few hundred
  environments (PPO on one device) to the throughput sizes of the reference's sweeps, for
  CartPole, Acrobot, the K-link pendulum (RK4 and semi-implicit Euler) and the C-legged body
  in both its arithmetics;
* one fused rollout of an evolution-strategies population on the caller's (P, D) weights
  (``rollout``): from the learner's default population to the reference's largest;
* one seeded generation (``generation``): the population regenerated from a seed, its
  rollout, the centred ranks, the update, and the greedy evaluation of the updated policy
  over 2,048 fresh episodes, as ``es.train`` runs them;
* populations early in training (most members fail at once and a few last) and late
  (``trained``: a policy that balances or stands, whose members run to the horizon).

Every result is a deterministic function of the inputs, bit for bit, so every tolerance is
"exact".
"""

import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "metal-rl-envs_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from hipenvs import (acrobot, acrobot_rollout, cartpole, cartpole_rollout, es, es_noise, legged,  # noqa: E402
                     legged_rollout, pendulum_aba)

EVAL_ENVS, EVAL_STEPS = 2048, 500   # es.evaluate's defaults
HIDDEN = (4, 8, 16, 32, 64)


# ---- the cases ----------------------------------------------------------------------------

def listed():
    return [
        # a learner's inner loop on a handful of environments: latency and the host path
        {"name": "cartpole_step_small", "kind": "step", "body": "cartpole", "n": 1000},
        # the largest batch of the throughput sweep, far beyond the caches
        {"name": "cartpole_step_large", "kind": "step", "body": "cartpole", "n": 1 << 24},
        # the reference's peak-rate shape for Acrobot
        {"name": "acrobot_step", "kind": "step", "body": "acrobot", "n": 262144},
        # the reference's pendulum benchmark: discrete torques, RK4, K = 16
        {"name": "aba_rk4_k16", "kind": "step", "body": "aba", "n": 65536, "k": 16, "euler": False, "wide": False},
        # long chains with continuous torques, semi-implicit Euler
        {"name": "aba_euler_k64", "kind": "step", "body": "aba", "n": 65536, "k": 64, "euler": True, "wide": False},
        # the quadruped under a learner with a couple of thousand environments
        {"name": "legged4_step_small", "kind": "step", "body": "legged", "n": 2048, "c": 4, "iters": 8,
         "assist": 0.0, "precision": "f32"},
        # the reference's price-list shape for the quadruped
        {"name": "legged4_step", "kind": "step", "body": "legged", "n": 65536, "c": 4, "iters": 8, "assist": 0.0,
         "precision": "f32"},
        # the reference's largest CartPole population, at the start of training
        {"name": "cartpole_rollout_large", "kind": "rollout", "body": "cartpole", "p": 262144, "hidden": 32,
         "horizon": 500, "sigma": 0.1, "trained": False},
        # the reference's Acrobot population
        {"name": "acrobot_rollout", "kind": "rollout", "body": "acrobot", "p": 4096, "hidden": 32, "horizon": 500,
         "sigma": 0.1, "trained": False},
        # the quadruped at full scale: 262,144 members, 64 hidden units, 1,000 steps
        {"name": "legged4_rollout_large", "kind": "rollout", "body": "legged", "p": 262144, "hidden": 64,
         "horizon": 1000, "sigma": 0.03, "trained": False, "c": 4, "iters": 8, "assist": 0.0},
        # a CartPole generation late in training, the population of the reference's benchmark
        {"name": "cartpole_generation", "kind": "generation", "body": "cartpole", "p": 4096, "hidden": 32,
         "horizon": 500, "sigma": 0.1, "trained": True},
        # a quadruped generation with the learner's defaults (population 1,024, 16 hidden units)
        {"name": "legged4_generation", "kind": "generation", "body": "legged", "p": 1024, "hidden": 16,
         "horizon": 500, "sigma": 0.1, "trained": True, "c": 4, "iters": 8, "assist": 0.0},
    ]


def _size(rng, lo, hi, even=False):
    """A whole number spread over the logarithm of [lo, hi]: now and then a power of two,
    otherwise anything, odd ones among them."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    n = 1 << int(round(math.log2(v))) if rng.random() < 0.2 else int(v)
    n = min(max(n, lo), hi)
    return n + (n & 1) if even else n


def draw(rng):
    kind = rng.choice(("step", "step", "rollout", "generation"))
    if kind == "step":
        body = rng.choice(("cartpole", "acrobot", "aba", "legged"))
        if body in ("cartpole", "acrobot"):
            return {"kind": kind, "body": body, "n": _size(rng, 256, 1 << 24 if body == "cartpole" else 1 << 21)}
        if body == "aba":
            return {"kind": kind, "body": body, "n": _size(rng, 256, 1 << 17), "k": rng.choice((1, 2, 3, 4, 8, 16, 32, 64)),
                    "euler": rng.random() < 0.5, "wide": rng.random() < 0.25}
        return {"kind": kind, "body": body, "n": _size(rng, 256, 1 << 18), "c": rng.choice((1, 2, 3, 4)),
                "iters": rng.choice((1, 4, 8, 16)), "assist": rng.choice((0.0, 0.0, 5.0)),
                "precision": rng.choice(("f32", "f32", "f32", "reference"))}
    body = rng.choice(("cartpole", "acrobot", "legged"))
    case = {"kind": kind, "body": body, "hidden": rng.choice(HIDDEN), "horizon": rng.randint(100, 500),
            "sigma": rng.choice((0.03, 0.1)), "trained": body != "acrobot" and rng.random() < 0.5}
    if body == "legged":
        case.update(c=rng.choice((1, 2, 3, 4)), iters=rng.choice((4, 8, 16)), assist=rng.choice((0.0, 0.0, 5.0)))
    # a trained population steps every member to the horizon, so its size is bounded to keep
    # its work below the full-scale quadruped's
    top = 1 << 18 if kind == "rollout" else 1 << 16
    if case["trained"] or body == "acrobot":
        top = 1 << 13 if body == "legged" else 1 << 16
    case["p"] = _size(rng, 256, top, even=True)
    return case


# ---- inputs -------------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 2654435761 % (1 << 62))
    return g


def _uniform(g, shape, lo, hi):
    return torch.rand(shape, generator=g, device="cuda") * (hi - lo) + lo


def _normal(g, shape, scale):
    return torch.randn(shape, generator=g, device="cuda") * scale


def _stand(c):
    """The legged body's standing pose (hip at the height of the innermost foot on the floor)."""
    angles = np.linspace(-0.25 * (c - 1), 0.25 * (c - 1), c) if c > 1 else np.zeros(1)
    q = np.concatenate([[0.0, math.cos(np.abs(angles).min()), 0.0], angles])
    return torch.tensor(np.concatenate([q, np.zeros_like(q)]).astype(np.float32), device="cuda")


def _policy_shape(case):
    if case["body"] == "legged":
        return 5 + 2 * case["c"], 3 * case["c"]
    return (4, 2) if case["body"] == "cartpole" else (6, 3)


def _theta(case, g):
    """The unperturbed policy (D,), in es.unflatten's layout: 0.1 N(0, 1), as training starts;
    trained, a balancing CartPole controller, or legs that pick zero torque and stand."""
    h, (i, o) = case["hidden"], _policy_shape(case)
    d = i * h + h + h * o + o
    theta = torch.randn(d, generator=g, device="cuda") * 0.1
    if not case["trained"]:
        return theta
    theta = theta * 0.2
    if case["body"] == "cartpole":
        gains = torch.tensor([0.1, 0.4, 4.0, 1.2], device="cuda")
        theta[:4 * h] += gains.repeat_interleave(h)               # every unit sees the same lean
        w2 = theta[5 * h:7 * h]
        w2[0::2] -= 1.0
        w2[1::2] += 1.0
    else:
        theta[d - o + 1::3] += 1.0                                # each leg's zero-torque head
    return theta


def _start(case, g, n):
    """Reset states of n members or environments."""
    if case["body"] == "legged":
        return _stand(case["c"])[:, None] + _uniform(g, (2 * (3 + case["c"]), n), -0.05, 0.05)
    bound = 0.05 if case["body"] == "cartpole" else 0.1
    return _uniform(g, (4, n), -bound, bound)


def _step_state(case, g):
    """A batch in mid-episode: spread over the states a running batch holds, some of them
    about to end their episode."""
    n, body = case["n"], case["body"]
    if body == "cartpole":
        return torch.stack([_normal(g, n, 0.6), _normal(g, n, 0.7), _uniform(g, n, -0.212, 0.212), _normal(g, n, 0.6)])
    if body == "acrobot":
        return torch.cat([_normal(g, (2, n), 1.0).clamp(-3.1, 3.1), _normal(g, (2, n), 2.0)])
    if body == "aba":
        k = case["k"]
        if case["wide"]:
            return torch.cat([_uniform(g, (k, n), -math.pi, math.pi), _uniform(g, (k, n), -3.0, 3.0)])
        return torch.cat([_uniform(g, (k, n), -0.2, 0.2), _normal(g, (k, n), 0.3)])
    c = case["c"]
    state = _stand(c)[:, None] + _uniform(g, (2 * (3 + c), n), -0.1, 0.1)
    state[1] += _uniform(g, n, -0.1, 0.1)
    state[2] += _normal(g, n, 0.2)
    state[3 + c:] += _normal(g, (3 + c, n), 0.5)
    return state


def prepare(case, seed):
    g = _gen(seed)
    s = {"case": case, "seed": int(seed) & 0x3FFFFFFF}
    if case["kind"] == "step":
        s["state"] = _step_state(case, g).contiguous()
        n, body = case["n"], case["body"]
        if body == "aba" and case["euler"]:
            s["action"] = _uniform(g, n, -1.0, 1.0)
        else:
            m = {"cartpole": 2, "acrobot": 3, "aba": 3}.get(body) or 3 ** case["c"]
            s["action"] = torch.randint(0, m, (n,), generator=g, device="cuda", dtype=torch.int32)
        if body == "aba":
            s["env"] = pendulum_aba.Pendulum(case["k"])
        elif body == "legged":
            s["env"] = legged.Legged(case["c"], case["iters"], case["precision"])
            if case["precision"] == "reference":
                s["state"] = s["state"].double()
        else:
            s["env"] = cartpole if body == "cartpole" else acrobot
        return s
    p = case["p"]
    theta = _theta(case, g)
    s["state"] = _start(case, g, p).contiguous()
    if case["kind"] == "rollout":
        half = torch.randn((p // 2, theta.shape[0]), generator=g, device="cuda")
        pop = torch.empty((p, theta.shape[0]), device="cuda")
        torch.add(theta, half, alpha=case["sigma"], out=pop[:p // 2])
        torch.add(theta, half, alpha=-case["sigma"], out=pop[p // 2:])
        s["theta_pop"] = pop
    else:
        s["theta"] = theta
        s["eval_state"] = _start(case, g, EVAL_ENVS).contiguous()
    return s


# ---- one pass -----------------------------------------------------------------------------

def _rollout_seeded(case, s):
    h, horizon, seed, sigma = case["hidden"], case["horizon"], s["seed"], case["sigma"]
    if case["body"] == "legged":
        return legged_rollout.rollout_seeded(s["state"], s["theta"], seed, sigma, h, horizon, case["c"],
                                             assist=case["assist"], iters=case["iters"])
    mod, sign = (cartpole_rollout, 1.0) if case["body"] == "cartpole" else (acrobot_rollout, -1.0)
    steps = mod.rollout_steps_seeded(s["state"], s["theta"], seed, sigma, h, horizon)
    return sign * steps, steps


def _evaluate(case, s, theta):
    if case["body"] == "legged":
        return legged_rollout.evaluate(s["eval_state"], theta, case["hidden"], EVAL_STEPS, case["c"], case["iters"])
    mod = cartpole_rollout if case["body"] == "cartpole" else acrobot_rollout
    return mod.evaluate(s["eval_state"], theta, case["hidden"], EVAL_STEPS)


def run(s):
    case = s["case"]
    if case["kind"] == "step":
        env = s["env"]
        env.reseed(s["seed"])  # the resets' counter: each pass steps the same step of the episode
        if case["body"] == "legged" and case["assist"]:
            return env.step(s["state"], s["action"], case["assist"])
        if case["body"] == "aba" and case["euler"]:
            return env.step_euler(s["state"], s["action"])
        return env.step(s["state"], s["action"])
    if case["kind"] == "rollout":
        if case["body"] == "legged":
            return legged_rollout.rollout(s["state"], s["theta_pop"], case["hidden"], case["horizon"], case["c"],
                                          assist=case["assist"], iters=case["iters"])
        mod = cartpole_rollout if case["body"] == "cartpole" else acrobot_rollout
        return mod.rollout_steps(s["state"], s["theta_pop"], case["hidden"], case["horizon"])
    fit, steps = _rollout_seeded(case, s)
    theta = es_noise.update(s["theta"], es.centered_ranks(fit), s["seed"], case["sigma"], 0.1)
    return {"fitness": fit, "steps": steps, "theta": theta, "scores": _evaluate(case, s, theta)}


# ---- what a pass cannot do without --------------------------------------------------------

def _legged_flops(c, iters, hidden=0):
    """Float operations of one control step (four substeps), counted from the equations: the
    mass matrix, its factor and 2C + 1 solves, the Delassus blocks, the sweeps; and the policy's."""
    n = 3 + c
    chol = n ** 3 // 3 + n * n
    substep = 30 * c + chol + (2 * c + 1) * 2 * n * n + 4 * c * c * 4 + 8 * c + iters * c * (8 * (c - 1) + 28) + n * (4 * c + 4)
    return 4 * substep + (hidden * (2 * (5 + 2 * c) + 2 * 3 * c) if hidden else 0)


def _step_flops(case):
    body, h = case["body"], case.get("hidden", 0)
    if body == "cartpole":
        return 26 + 12 * h
    if body == "acrobot":
        return 202 + 18 * h
    if body == "aba":
        return case["k"] * (110 * (1 if case["euler"] else 4) + 12)
    return _legged_flops(case["c"], case["iters"], h)


def _mean_steps(case):
    """Steps a member takes on average: a few before an untrained member fails (about 15 for
    CartPole, 40 for the legged bodies), nearly the horizon for Acrobot and trained members."""
    if case["trained"] or case["body"] == "acrobot":
        return case["horizon"]
    return min(case["horizon"], 15 if case["body"] == "cartpole" else 40)


def work(case):
    if case["kind"] == "step":
        body = case["body"]
        rows = 4 if body in ("cartpole", "acrobot") else 2 * case["k"] if body == "aba" else 2 * (3 + case["c"])
        width = 8 if case.get("precision") == "reference" else 4
        return {"bytes": case["n"] * (2 * rows * width + 9), "flops": case["n"] * _step_flops(case)}
    i, o = _policy_shape(case)
    h, p = case["hidden"], case["p"]
    d = i * h + h + h * o + o
    rows = 2 * (3 + case["c"]) if case["body"] == "legged" else 4
    outs = 2 if case["body"] == "legged" else 1
    flops = p * _mean_steps(case) * _step_flops(case)
    if case["kind"] == "rollout":
        return {"bytes": 4 * p * (d + rows + outs), "flops": flops}
    evaluated = EVAL_ENVS * (EVAL_STEPS if case["trained"] or case["body"] == "acrobot" else 40) * _step_flops(case)
    noise = 2 * (p // 2) * d * 30  # drawn for the rollout and again for the update
    return {"bytes": 4 * (p * (rows + 3) + 3 * d + EVAL_ENVS * (rows + 1)), "flops": flops + evaluated + noise}


def tolerance(case):
    """Every path fixes the order and rounding of its operations, so two correct builds agree
    bit for bit."""
    return "exact"


# ---- the same results in 64 bits ------------------------------------------------------------
# The equations of each body in float64 torch, from the inputs of prepare(). Rollouts are not
# restated: an episode's length is decided by thresholds and argmaxes along a trajectory that
# amplifies rounding, and has no 64-bit value to be near to, but for CartPole's, whose pole
# either falls at once or is held.

_GOLDEN, _M32 = 0x9E3779B9, 0xFFFFFFFF


def _pcg(v):
    """The PCG hash on uint32 values held in int64."""
    s = (v * 747796405 + 2891336453) & _M32
    w = (((s >> ((s >> 28) + 4)) ^ s) * 277803737) & _M32
    return (w >> 22) ^ w


def _fresh(seed, n, offsets, bound):
    """The reset draws of step counter `seed`: row r of env e from hash(seed ^ e golden + offset_r)."""
    e = torch.arange(n, dtype=torch.int64, device="cuda")
    h = (seed & _M32) ^ ((e * _GOLDEN) & _M32)
    rows = [(_pcg((h + o) & _M32) >> 8).double() * 2.0 ** -23 - 1.0 for o in offsets]
    return torch.stack(rows) * bound


_FOUR = (0, 0x85EBCA6B, 0xC2B2AE35, 0x27D4EB2F)


def _strided(rows):
    return [(r * 0x85EBCA6B) & _M32 for r in range(rows)]


def _wrap(x):
    return x - 2 * math.pi * torch.floor((x + math.pi) / (2 * math.pi))


def _cartpole64(s, push):
    x, xd, th, thd = s
    sin, cos = torch.sin(th), torch.cos(th)
    temp = (torch.where(push, 10.0, -10.0).double() + 0.05 * thd * thd * sin) / 1.1
    tha = (9.8 * sin - cos * temp) / (0.5 * (4.0 / 3.0 - 0.1 * cos * cos / 1.1))
    xa = temp - 0.05 * tha * cos / 1.1
    out = torch.stack([x + 0.02 * xd, xd + 0.02 * xa, th + 0.02 * thd, thd + 0.02 * tha])
    return out, (out[0].abs() > 2.4) | (out[2].abs() > 12 * 2 * math.pi / 360)


def _acrobot64(s, torque):
    def rate(s):
        a, b, da, db = s
        c2, s2 = torch.cos(b), torch.sin(b)
        d1 = 0.25 + (1.25 + c2) + 2.0
        d2 = 0.25 + 0.5 * c2 + 1.0
        phi2 = 4.9 * torch.cos(a + b - math.pi / 2)
        phi1 = -0.5 * db * db * s2 - db * da * s2 + 14.7 * torch.cos(a - math.pi / 2) + phi2
        ddb = (torque + d2 / d1 * phi1 - 0.5 * da * da * s2 - phi2) / (1.25 - d2 * d2 / d1)
        return torch.stack([da, db, -(d2 * ddb + phi1) / d1, ddb])

    k1 = rate(s)
    k2 = rate(s + 0.1 * k1)
    k3 = rate(s + 0.1 * k2)
    k4 = rate(s + 0.2 * k3)
    n = s + 0.2 / 6 * (k1 + 2 * k2 + 2 * k3 + k4)
    n = torch.stack([_wrap(n[0]), _wrap(n[1]), n[2].clamp(-4 * math.pi, 4 * math.pi), n[3].clamp(-9 * math.pi, 9 * math.pi)])
    return n, -torch.cos(n[0]) - torch.cos(n[0] + n[1]) > 1.0


def _chain64(th, om, torque):
    """Accelerations of a hanging chain of K unit masses on unit rods: with absolute angles,
    M_ij = (K - max(i, j)) cos(th_i - th_j), solved densely env by env."""
    k = th.shape[0]
    idx = torch.arange(k, device=th.device)
    mu = (k - torch.maximum(idx[:, None], idx[None, :])).double()
    out = torch.empty_like(th)
    for lo in range(0, th.shape[1], 8192):
        t, o = th[:, lo:lo + 8192].T, om[:, lo:lo + 8192].T
        diff = t[:, :, None] - t[:, None, :]
        rhs = -(mu * torch.sin(diff) * (o * o)[:, None, :]).sum(2) - 9.8 * torch.diagonal(mu) * torch.sin(t)
        rhs[:, 0] += torque[lo:lo + 8192]
        out[:, lo:lo + 8192] = torch.linalg.solve(mu * torch.cos(diff), rhs).T
    return out


def _aba64(s, action, k, euler):
    th, om = s[:k], s[k:]
    if euler:
        om2 = om + 0.01 * _chain64(th, om, action.double())
        th2 = th + 0.01 * om2
    else:
        torque = (action - 1).double()

        def rate(y):
            return torch.cat([y[k:], _chain64(y[:k], y[k:], torque)])

        k1 = rate(s)
        k2 = rate(s + 0.01 * k1)
        k3 = rate(s + 0.01 * k2)
        k4 = rate(s + 0.02 * k3)
        n = s + 0.02 / 6 * (k1 + 2 * k2 + 2 * k3 + k4)
        th2, om2 = n[:k], n[k:]
    n = torch.cat([_wrap(th2), om2.clamp(-10 * math.pi, 10 * math.pi)])
    return n, -torch.cos(n[:k]).sum(0) > k / 2


def _legged64(s, action, c, iters, assist):
    """Four substeps: M = diag(1, 1, 0.1) + 0.2 sum J^T J, the free velocity, and `iters` sweeps
    of projected Gauss-Seidel with the exact 2x2 contact solve, friction 0.7."""
    d = 3 + c
    q, v = s[:d].T.clone(), s[d:].T.clone()
    m = q.shape[0]
    for _ in range(4):
        eye = torch.zeros((m, d, d), dtype=torch.float64, device=q.device)
        eye[:, 0, 0] = eye[:, 1, 1] = 1.0
        eye[:, 2, 2] = 0.1
        jac, drift = [], torch.zeros((m, d), dtype=torch.float64, device=q.device)
        mass = eye
        for k in range(c):
            a, ad = q[:, 2] + q[:, 3 + k], v[:, 2] + v[:, 3 + k]
            j = torch.zeros((m, 2, d), dtype=torch.float64, device=q.device)
            j[:, 0, 0] = j[:, 1, 1] = 1.0
            for row, f in ((0, torch.cos(a)), (1, torch.sin(a))):
                j[:, row, 2] = j[:, row, 3 + k] = f
            jac.append(j)
            acc = torch.stack([-torch.sin(a) * ad * ad, torch.cos(a) * ad * ad + 9.8], 1)
            drift += 0.2 * (j.transpose(1, 2) @ acc[:, :, None]).squeeze(2)
            mass = mass + 0.2 * (j.transpose(1, 2).contiguous() @ j)
        force = -drift
        force[:, 1] -= 9.8
        for k in range(c):
            force[:, 3 + k] += ((action // 3 ** k) % 3 - 1).double() * 2.0
        force[:, 2] -= assist * q[:, 2] + 0.1 * assist * v[:, 2]
        inv = torch.linalg.inv(mass)
        free = v + 0.01 * (inv @ force[:, :, None]).squeeze(2)
        big = torch.cat(jac, 1)                                   # (m, 2c, d)
        resp = inv @ big.transpose(1, 2).contiguous()             # (m, d, 2c)
        delassus = big @ resp
        w0 = (big @ free[:, :, None]).squeeze(2)
        lam = torch.zeros((m, 2 * c), dtype=torch.float64, device=q.device)
        for _ in range(iters):
            for k in range(c):
                own = delassus[:, 2 * k:2 * k + 2, 2 * k:2 * k + 2]
                w = w0[:, 2 * k:2 * k + 2] + (delassus[:, 2 * k:2 * k + 2] @ lam[:, :, None]).squeeze(2)
                w = w - (own @ lam[:, 2 * k:2 * k + 2, None]).squeeze(2)
                wt, wn = w[:, 0], w[:, 1]
                tt, tn, nn = own[:, 0, 0], own[:, 0, 1], own[:, 1, 1]
                depth = -(q[:, 1] - torch.cos(q[:, 2] + q[:, 3 + k]))
                gap = 20.0 * depth.clamp(min=0.0) - wn
                det = tt * nn - tn * tn
                ln_s, lt_s = (tt * gap + tn * wt) / det, (-nn * wt - tn * gap) / det
                up, um = nn + 0.7 * tn, nn - 0.7 * tn
                ln_p = torch.where(up > 0, (gap / up).clamp(min=0.0), 0.0)
                ln_m = torch.where(um > 0, (gap / um).clamp(min=0.0), 0.0)
                plus = wt + (tt * 0.7 + tn) * ln_p <= 0
                stick = lt_s.abs() <= 0.7 * ln_s
                ln = torch.where(stick, ln_s, torch.where(plus, ln_p, ln_m))
                lt = torch.where(stick, lt_s, torch.where(plus, 0.7 * ln_p, -0.7 * ln_m))
                on = (depth >= 0) & (ln > 0) & (gap > 0)
                lam[:, 2 * k] = torch.where(on, lt, 0.0)
                lam[:, 2 * k + 1] = torch.where(on, ln, 0.0)
        v = free + (resp @ lam[:, :, None]).squeeze(2)
        q = q + 0.01 * v
    n = torch.cat([q, v], 1).T
    return n, (n[1] < 0.6) | (n[2].abs() > 1.0)


def _cartpole_rollout64(case, s):
    h, p = case["hidden"], case["p"]
    theta, state = s["theta_pop"], s["state"].double()
    alive = torch.arange(p, device="cuda")
    steps = torch.zeros(p, dtype=torch.float64, device="cuda")
    w = theta.double()
    for _ in range(case["horizon"]):
        if not alive.numel():
            break
        hid = torch.tanh((state.T[:, :, None] * w[:, :4 * h].view(-1, 4, h)).sum(1) + w[:, 4 * h:5 * h])
        out = (hid[:, :, None] * w[:, 5 * h:7 * h].view(-1, h, 2)).sum(1) + w[:, 7 * h:]
        state, done = _cartpole64(state, out[:, 1] > out[:, 0])
        keep = ~done
        steps[alive[keep]] += 1
        if done.any():
            alive, state, w = alive[keep], state[:, keep], w[keep]
    return steps


def exact(case, seed):
    if case["kind"] == "rollout" and case["body"] == "cartpole" and not case["trained"]:
        return _cartpole_rollout64(case, prepare(case, seed))
    if case["kind"] != "step":
        return None
    s = prepare(case, seed)
    state, action, n, body = s["state"].double(), s["action"], case["n"], case["body"]
    counter = s["seed"] + 1  # step() pre-increments the counter that reseed() set
    if body == "cartpole":
        out, done = _cartpole64(state, action == 1)
        fresh, reward = _fresh(counter, n, _FOUR, 0.05), torch.ones(n, dtype=torch.float64, device="cuda")
    elif body == "acrobot":
        out, done = _acrobot64(state, (action - 1).double())
        fresh, reward = _fresh(counter, n, _FOUR, 0.1), -(~done).double()
    elif body == "aba":
        k = case["k"]
        out, done = _aba64(state, action, k, case["euler"])
        fresh, reward = _fresh(counter, n, _strided(2 * k), 0.1), -(~done).double()
        if case["euler"]:
            fresh[k:] = 0.0
    else:
        c = case["c"]
        out, done = _legged64(state, action, c, case["iters"], case["assist"])
        fresh = _stand(c).double()[:, None] + _fresh(counter, n, _strided(2 * (3 + c)), 0.05)
        reward = torch.where(done, 0.0, out[3 + c] + 1.0)
    return torch.where(done[None], fresh, out), reward, None
