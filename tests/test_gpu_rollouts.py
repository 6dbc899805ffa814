"""Fused ES rollout kernels vs the oracle, through the C ABI (GPU).

Bar: bit-exact fitness for every member. The oracle's fused-rollout restatement
is itself checked against its es.loop_fitness restatement (test_oracle_es.py),
which is the reference's test_es.py:46-69 gate made exact.
"""

import numpy as np
import pytest
import torch

from oracle import acrobot as oa
from oracle import cartpole as oc
from oracle import es as oes

pytestmark = pytest.mark.gpu


def to_np(t):
    return t.detach().cpu().numpy()


def population(p, d, seed, scale=None, sigma=0.1):
    """theta_pop: scale * N(0,1) rows, or (scale None) the antithetic ES population
    theta0 + sigma * [half; -half] around theta0 = 0.1 * N(0, 1)."""
    r = np.random.default_rng(seed)
    if scale is not None:
        return (r.standard_normal((p, d)) * scale).astype(np.float32)
    theta0 = (r.standard_normal(d) * 0.1).astype(np.float32)
    half = r.standard_normal((p // 2, d)).astype(np.float32)
    eps = np.concatenate([half, -half])
    return (theta0[None, :] + np.float32(sigma) * eps).astype(np.float32)


@pytest.mark.parametrize("hidden", [4, 8, 16, 32, 64])
def test_cartpole_rollout_matches_oracle(dev, hidden):
    from hipenvs import cartpole_rollout

    p, horizon = 512, 200
    theta = population(p, 7 * hidden + 2, hidden, scale=0.5)
    state = oc.reset(p, seed=3)
    got = cartpole_rollout.rollout_steps(torch.from_numpy(state).to(dev), torch.from_numpy(theta).to(dev), hidden, horizon)
    np.testing.assert_array_equal(to_np(got), oc.rollout_survived(state, theta, hidden, horizon))


@pytest.mark.parametrize("hidden", [4, 8, 16, 32, 64])
def test_acrobot_rollout_matches_oracle(dev, hidden):
    from hipenvs import acrobot_rollout

    p, horizon = 512, 120
    theta = population(p, 10 * hidden + 3, hidden, scale=0.5)
    state = oa.reset(p, seed=4)
    got = acrobot_rollout.rollout_steps(torch.from_numpy(state).to(dev), torch.from_numpy(theta).to(dev), hidden, horizon)
    np.testing.assert_array_equal(to_np(got), oa.rollout_steps(state, theta, hidden, horizon))


@pytest.mark.parametrize("hidden", [8, 32])
def test_large_populations_one_member_per_lane(dev, hidden):
    """Populations past the 4-lane form's bound start with one lane per member; both bodies, bit for
    bit against the oracle."""
    from hipenvs import acrobot_rollout, cartpole_rollout

    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    p = (256 if hidden >= 16 else 128) * cus + 1
    theta = population(p, 7 * hidden + 2, 100 + hidden, scale=0.5)
    state = oc.reset(p, seed=5)
    got = cartpole_rollout.rollout_steps(torch.from_numpy(state).to(dev), torch.from_numpy(theta).to(dev), hidden, 150)
    np.testing.assert_array_equal(to_np(got), oc.rollout_survived(state, theta, hidden, 150))
    p = 128 * cus + 1
    theta = population(p, 10 * hidden + 3, 200 + hidden, scale=0.5)
    state = oa.reset(p, seed=6)
    got = acrobot_rollout.rollout_steps(torch.from_numpy(state).to(dev), torch.from_numpy(theta).to(dev), hidden, 60)
    np.testing.assert_array_equal(to_np(got), oa.rollout_steps(state, theta, hidden, 60))


def _mixed_population(body, p, hidden, seed):
    """(theta, state, horizon) of members that end at many different steps, so that a wave passes
    through its lane-group forms in mid-episode. CartPole: wild policies, of which one in twelve
    balances. Acrobot: wild policies from fast start states, most of which swing past the goal's
    height sooner or later (from rest hardly any does)."""
    i, o = (4, 2) if body == "cartpole" else (6, 3)
    r = np.random.default_rng(seed)
    theta = (r.standard_normal((p, i * hidden + hidden + hidden * o + o)) * 0.3).astype(np.float32)
    if body == "acrobot":
        state = np.stack([r.uniform(-np.pi, np.pi, p), r.uniform(-np.pi, np.pi, p), r.normal(0, 6, p),
                          r.normal(0, 12, p)]).astype(np.float32)
        return theta, state, 90
    good = r.random(p) < 1 / 12
    theta[good] *= np.float32(0.2)
    theta[good, :4 * hidden] += np.repeat(np.array([0.1, 0.4, 4.0, 1.2], np.float32), hidden)
    theta[good, 5 * hidden:7 * hidden:2] -= np.float32(1.0)
    theta[good, 5 * hidden + 1:7 * hidden:2] += np.float32(1.0)
    return theta, oc.reset(p, seed=11), 150


def _share_narrowing(scores, horizon, members, left):
    """Of the blocks of `members` consecutive scores (a wave's members), the share that comes down to
    `left` live ones after the first step and before the horizon."""
    s = np.sort(scores[:len(scores) // members * members].reshape(-1, members), axis=1)
    at = s[:, members - left - 1]  # the step that ends all but the `left` longest
    return ((at > 0) & (at < horizon)).mean()


# members per CU at which the starting form changes (16, 4, 1 lanes per member), per body and H
_FORM_BOUNDS = {("cartpole", 4): (32, 128), ("cartpole", 32): (32, 256), ("cartpole", 64): (32, None),
                ("acrobot", 8): (16, 128), ("acrobot", 32): (16, 128), ("acrobot", 64): (16, None)}


@pytest.mark.parametrize("body,hidden", sorted(_FORM_BOUNDS))
def test_every_starting_form_gives_the_same_scores(dev, body, hidden):
    """Populations just past each bound of the launch rule (ragged last waves) against the same
    members run in slices small enough for the 16-lane form, which the tests above pin to the
    oracle: every member's score equal, whatever forms its wave went through. Nearly every wave
    regroups in mid-episode: from one lane at 16 members left, from 4 lanes at 4."""
    from hipenvs import acrobot_rollout, cartpole_rollout

    mod = cartpole_rollout if body == "cartpole" else acrobot_rollout
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    b16, b4 = _FORM_BOUNDS[body, hidden]
    p = (b4 or 2 * b16) * cus + 37
    theta, state, horizon = _mixed_population(body, p, hidden, 7 + hidden)
    theta, state = torch.from_numpy(theta).to(dev), torch.from_numpy(state).to(dev)
    want = torch.cat([mod.rollout_steps(state[:, a:a + 4001].contiguous(), theta[a:a + 4001], hidden, horizon)
                      for a in range(0, p, 4001)])
    for n in (p, b16 * cus + 1, b16 * cus):
        got = mod.rollout_steps(state[:, :n].contiguous(), theta[:n], hidden, horizon)
        assert torch.equal(got, want[:n]), n
    scores = to_np(want)
    assert len(np.unique(scores)) > 40
    for members, left, share in ((64, 16, 0.9), (16, 4, 0.9), (64, 4, 0.15)):  # of waves: measured 1, 0.98, 0.25
        assert _share_narrowing(scores, horizon, members, left) > share, (members, left)
    one = mod.rollout_steps(state[:, :1].contiguous(), theta[:1], hidden, horizon)
    assert torch.equal(one, want[:1])
    for h in (0, 1):  # nothing to step; the horizon reached in the first form
        got = mod.rollout_steps(state, theta, hidden, h)
        assert torch.equal(got, torch.clamp(want, max=h))


def test_shared_policy_takes_every_starting_form(dev):
    """The greedy evaluation (member stride 0) past the lane-group bounds equals its slices."""
    from hipenvs import acrobot_rollout, cartpole_rollout

    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    n = 130 * cus + 3
    for mod, reset, d in ((cartpole_rollout, oc.reset, 7 * 8 + 2), (acrobot_rollout, oa.reset, 10 * 8 + 3)):
        theta = torch.from_numpy(population(2, d, 3, scale=0.4)[0]).to(dev)
        state = torch.from_numpy(reset(n, seed=2)).to(dev)
        got = mod.evaluate(state, theta, 8, 80)
        want = torch.cat([mod.evaluate(state[:, a:a + 4000].contiguous(), theta, 8, 80) for a in range(0, n, 4000)])
        assert torch.equal(got, want)


def test_shared_policy_past_2_to_the_30_envs(dev):
    """At H = 64 an evaluation runs 4 lanes per env; one of more than 2^30 envs (21 GB of states and
    scores) needs more threads than a grid's x can have."""
    from hipenvs import cartpole_rollout

    block, n = 1 << 20, (1 << 30) + 17
    part = oc.reset(block, seed=6)
    part[2, ::5] = 0.207  # these fall within the two steps
    part[3, ::5] = 0.2
    part = torch.from_numpy(part).to(dev)
    state = torch.empty((4, n), dtype=torch.float32, device=dev)
    for a in range(0, n, block):
        state[:, a:a + block] = part[:, :n - a]
    theta = torch.from_numpy(population(2, 7 * 64 + 2, 3, scale=0.4)[0]).to(dev)
    want = cartpole_rollout.evaluate(part, theta, 64, 2)
    assert len(want.unique()) > 1
    got = cartpole_rollout.evaluate(state, theta, 64, 2)
    del state
    assert torch.equal(got[1 << 30:], want[:17])
    for a in range(0, 1 << 30, 1 << 28):
        assert bool((got[a:a + (1 << 28)].view(-1, block) == want).all())


def test_config2_cartpole_population(dev):
    """P = 4,096 antithetic members (sigma 0.1) around theta0 = 0.1 N(0,1), H = 32, horizon 500."""
    from hipenvs import cartpole_rollout

    p, hidden, horizon = 4096, 32, 500
    theta = population(p, 7 * hidden + 2, 0)
    state = oc.reset(p, seed=0)
    got = to_np(cartpole_rollout.rollout_steps(torch.from_numpy(state).to(dev), torch.from_numpy(theta).to(dev),
                                               hidden, horizon))
    np.testing.assert_array_equal(got, oc.rollout_survived(state, theta, hidden, horizon))


def test_config2_acrobot_population(dev):
    from hipenvs import acrobot_rollout

    p, hidden, horizon = 4096, 32, 500
    theta = population(p, 10 * hidden + 3, 1)
    state = oa.reset(p, seed=0)
    got = to_np(acrobot_rollout.rollout_steps(torch.from_numpy(state).to(dev), torch.from_numpy(theta).to(dev),
                                              hidden, horizon))
    np.testing.assert_array_equal(got, oa.rollout_steps(state, theta, hidden, horizon))


def test_rollout_edge_cases(dev):
    """Horizon 0, a single member, a population that is not a multiple of the wave size."""
    from hipenvs import cartpole_rollout

    for p, horizon in ((1, 50), (65, 0), (130, 7)):
        theta = population(p, 7 * 8 + 2, p, scale=1.0)
        state = oc.reset(p, seed=p)
        got = cartpole_rollout.rollout_steps(torch.from_numpy(state).to(dev), torch.from_numpy(theta).to(dev), 8, horizon)
        np.testing.assert_array_equal(to_np(got), oc.rollout_survived(state, theta, 8, horizon))


def test_unsupported_hidden_raises(dev):
    from hipenvs import cartpole_rollout

    with pytest.raises(ValueError):
        cartpole_rollout.rollout_steps(torch.zeros((4, 8), device=dev), torch.zeros((8, 7 * 5 + 2), device=dev), 5, 10)
