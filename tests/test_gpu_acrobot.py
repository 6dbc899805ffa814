"""Acrobot HIP step kernel vs the oracle, through the C ABI (GPU). Bar: bit-exact."""

import numpy as np
import pytest
import torch

from oracle import acrobot as oa
from oracle import rng
from test_oracle_acrobot import random_batch

pytestmark = pytest.mark.gpu


def to_np(t):
    return t.detach().cpu().numpy()


@pytest.mark.parametrize("n", [1, 200, 4096, 5000])
def test_step_matches_oracle_on_random_states(dev, n):
    """test_acrobot.py:98-122's random states, every column compared (terminal ones too)."""
    from hipenvs import acrobot

    state, action = random_batch(n, seed=n)
    acrobot.reseed(10)
    ns, rew, done = acrobot.step(torch.from_numpy(state).to(dev), torch.from_numpy(action).to(dev))
    ens, erew, edone = oa.step(state, action, seed=11)
    np.testing.assert_array_equal(to_np(ns), ens)
    np.testing.assert_array_equal(to_np(rew), erew)
    np.testing.assert_array_equal(to_np(done), edone)


def test_step_bit_exact_at_the_benchmark_size(dev):
    """N = 262,144, the reference's Acrobot step benchmark shape, with mixed terminations."""
    from hipenvs import acrobot

    state, action = random_batch(1 << 18, seed=18)
    acrobot.reseed(30)
    ns, rew, done = acrobot.step(torch.from_numpy(state).to(dev), torch.from_numpy(action).to(dev))
    ens, erew, edone = oa.step(state, action, seed=31)
    np.testing.assert_array_equal(to_np(done), edone)
    np.testing.assert_array_equal(to_np(ns), ens)
    np.testing.assert_array_equal(to_np(rew), erew)
    assert 0 < edone.sum() < len(edone)


def _far_states(n, seed):
    """random_batch with theta2 of 1e18 to 1e20: det_sincos's reduction has no digits left there and
    its cosine, which the mass matrix is a function of, takes any size; past 4e19 the square of
    an entry overflows, and the results stay finite."""
    state, action = random_batch(n, seed=seed)
    r = np.random.default_rng(seed + 1)
    state[1] = (10.0 ** r.uniform(18, 20, n) * r.choice([-1, 1], n)).astype(np.float32)
    assert (np.abs(oa.detmath.cos(state[1])) > 4e19).sum() > n // 4
    return state, action


def test_step_with_angles_past_the_sincos_reduction(dev):
    from hipenvs import acrobot

    state, action = _far_states(5000, seed=40)
    with np.errstate(all="ignore"):
        want = oa.step(state, action, seed=11)
    assert np.isfinite(want[0]).all()
    acrobot.reseed(10)
    got = acrobot.step(torch.from_numpy(state).to(dev), torch.from_numpy(action).to(dev))
    for g, w in zip(got, want):
        np.testing.assert_array_equal(to_np(g), w)


def test_rollout_with_angles_past_the_sincos_reduction(dev):
    """The same start states in the rollout, in its 16-, 4- and 1-lane forms: five steps, of which
    the first is out of range (angles are wrapped after it)."""
    from hipenvs import acrobot_rollout

    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    n = 128 * cus + 1
    state, _ = _far_states(n, seed=41)
    theta = (np.random.default_rng(5).standard_normal((n, 10 * 8 + 3)) * 0.5).astype(np.float32)
    with np.errstate(all="ignore"):
        want = oa.rollout_steps(state, theta, 8, 5)
    assert len(np.unique(want)) > 3
    dstate, dtheta = torch.from_numpy(state).to(dev), torch.from_numpy(theta).to(dev)
    for m in (n, 128 * cus, 16 * cus):
        got = acrobot_rollout.rollout_steps(dstate[:, :m].contiguous(), dtheta[:m], 8, 5)
        np.testing.assert_array_equal(to_np(got), want[:m])


def test_reset_matches_counter_rng(dev):
    from hipenvs import acrobot

    np.testing.assert_array_equal(to_np(acrobot.reset(3000, seed=4, device=dev)), oa.reset(3000, seed=4))


def test_teacher_forced_and_free_running_chains(dev):
    """300 teacher-forced steps (each step from the oracle's state) then 100 free-running
    steps with identical done flags at every step."""
    from hipenvs import acrobot

    n = 4096
    state = oa.reset(n, seed=0)
    acrobot.reseed(0)
    for t in range(1, 301):
        a = rng.uniform_actions(t, n, 3)
        ns, _, done = acrobot.step(torch.from_numpy(state).to(dev), torch.from_numpy(a).to(dev))
        ens, _, edone = oa.step(state, a, seed=t)
        assert np.array_equal(to_np(ns), ens) and np.array_equal(to_np(done), edone), f"step {t}"
        state = ens
    s_dev = torch.from_numpy(state).to(dev)
    for t in range(301, 401):
        a = rng.uniform_actions(t, n, 3)
        s_dev, _, d_dev = acrobot.step(s_dev, torch.from_numpy(a).to(dev))
        state, _, d_ref = oa.step(state, a, seed=t)
        np.testing.assert_array_equal(to_np(d_dev), d_ref, err_msg=f"step {t}")
    np.testing.assert_array_equal(to_np(s_dev), state)


def test_resets_and_lazy_chain(dev):
    """test_acrobot.py:125-146 on the device."""
    from hipenvs import acrobot

    n = 4096
    terminal = torch.zeros((4, n), device=dev)
    terminal[0] = np.pi
    ones = torch.ones(n, dtype=torch.int32, device=dev)
    first = to_np(acrobot.step(terminal, ones)[0])
    second = to_np(acrobot.step(terminal, ones)[0])
    assert np.all(np.abs(first) <= oa.RESET_BOUND) and not np.allclose(first, second)
    assert abs(first.std() - oa.RESET_BOUND / np.sqrt(3)) < 0.002
    state = acrobot.reset(n, device=dev)
    for t in range(100):
        state, _, _ = acrobot.step(state, torch.randint(0, 3, (n,), device=dev, dtype=torch.int32))
    out = to_np(state)
    assert np.isfinite(out).all() and np.all(np.abs(out[:2]) <= np.pi)
