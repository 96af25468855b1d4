"""Observation and head widths that no built-in env has (tests/envs/ramp.h), odd
ones among them, through every collect and forward kernel that pairs, pads or
stages operands by width: the env side of a collect against a rollout of the
same actions, bit for bit, the policy side against a float64 network."""
import ctypes
import os

import numpy as np
import pytest

from parity import assert_bit_exact
from test_gpu_nonfinite import network

pytestmark = pytest.mark.gpu

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "envs", "build", "libmg_test_envs.so")
WIDTHS = {"ramp1": (1, 2), "ramp3": (3, 4), "ramp15": (15, 15), "ramp33": (33, 7), "ramp63": (63, 15)}


@pytest.fixture(scope="module")
def ramps(mg):
    assert os.path.exists(LIB), f"{LIB} missing: run __graft_entry__.build()"
    ctypes.CDLL(LIB)
    return mg


def policy(mg, gym, T, layers, scale):
    model = mg.PPOModel(gym, horizon=T, minibatch=64, layers=layers, scale=scale)
    pv, P, rs = model.pv, model.params(), np.random.default_rng(1)
    P[pv.off_in_b:pv.off_in_b + 128] = 0.3 * rs.standard_normal(128)  # a row of one float is a line
    P[pv.off_head:pv.off_head + 128 * pv.head_dim] += 0.1 * rs.standard_normal(128 * pv.head_dim)
    model.set_params(P)
    return model, P


@pytest.mark.parametrize("env", sorted(WIDTHS))
# 16-row tiles, 32-row ones (ramp15: its head is wide), two shares, one, and past 32 floats
@pytest.mark.parametrize("n", [64, 8192, 8256, 16448, 32832])
@pytest.mark.parametrize("layers,scale", [(2, 2), (2, 4), (1, 1)])
def test_collect(ramps, env, n, layers, scale):
    mg, (O, A), T = ramps, WIDTHS[env], 3
    gym, twin = (mg.Gym("rollout_test_" + env, n, 2) for _ in range(2))
    assert (gym.obs_dim, gym.act_dim) == (O, A)
    model, P = policy(mg, gym, T, layers, scale)
    model.collect()
    s = model.download_slots()
    # the first collect steps every env once with action 0 before the horizon
    actions = np.concatenate([np.zeros((1, n), np.int32), s["actions"]])
    assert ((actions >= 0) & (actions < A)).all()
    want = network(model.pv, P, s["obs"].reshape(-1, O), np.float64).reshape(T + 1, n, A + 1)
    np.testing.assert_allclose(model.head(), want[T], rtol=0, atol=1e-4)
    np.testing.assert_allclose(s["value"], want[:T, :, A], rtol=0, atol=1e-4)
    z = want[:T, :, :A]
    z = z - z.max(-1, keepdims=True)
    logp = np.take_along_axis(z - np.log(np.exp(z).sum(-1, keepdims=True)), s["actions"][..., None], -1)[..., 0]
    np.testing.assert_allclose(s["logp"], logp, rtol=0, atol=1e-4)
    # an env's generator also draws its actions, so a rollout of them follows until the first reset
    _, obs, rew, dn = twin.rollout_given(T + 1, actions)
    obs, dn = obs.download(np.float32, (T + 1, n, O)), dn.download(np.uint8, (T + 1, n))
    rew = rew.download(np.float32, (T + 1, n))
    alive = np.concatenate([np.ones((1, n), bool), np.cumsum(dn, 0)[:T] == 0])
    assert alive[T].mean() > 0.3
    assert_bit_exact(s["obs"][alive], obs[alive], "obs")
    assert_bit_exact(s["reward"][alive[1:]], rew[1:][alive[1:]], "reward")
    assert_bit_exact(s["done"][alive[1:]], dn[1:][alive[1:]], "done")


@pytest.mark.parametrize("env", sorted(WIDTHS))
@pytest.mark.parametrize("rows", [33, 4096, 4097, 8200])  # 4097: past 8 columns the 32-row tiles
def test_forward(ramps, env, rows):
    mg, (O, A) = ramps, WIDTHS[env]
    model, P = policy(mg, mg.Gym("rollout_test_" + env, 64, 0), 1, 3, 3)
    obs = np.random.default_rng(0).normal(0, 1.5, (rows, O)).astype(np.float32)
    np.testing.assert_allclose(model.forward(obs), network(model.pv, P, obs, np.float64), rtol=0, atol=1e-4)
