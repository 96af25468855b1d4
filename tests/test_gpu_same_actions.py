"""The fp32 tiles' arithmetic that the collects on binary16 pairs repeat for a
draw near an edge of the CDF: the heads of single rows bit for bit, and the
actions of whole collects. The tiles themselves run from a view without the
planes of pairs (mg_policy_view)."""
import ctypes
import os

import numpy as np
import pytest

from parity import ENVS, assert_bit_exact
from test_gpu_policy_view import collect_with_view

pytestmark = pytest.mark.gpu

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "envs", "build", "libmg_test_envs.so")


def without_planes(pv):
    view = type(pv)()
    ctypes.pointer(view)[0] = pv
    view.frag_fwd32_bf = view.frag_fwd16_bf = None
    return view


def both(mg, env, n, T, layers, scale, head):
    """One collect from the same envs by the library's kernel and by the tiles;
    head: a factor on the policy head's weights."""
    gym = mg.Gym(ENVS[env][1], n, 4)
    model = mg.PPOModel(gym, horizon=T, minibatch=64, layers=layers, scale=scale, seed=4)
    pv, P, rs = model.pv, model.params(), np.random.default_rng(7)
    for l in range(layers + 1):
        P[pv.off_ln_gamma[l]:pv.off_ln_gamma[l] + 128] = 1 + 0.1 * rs.standard_normal(128)
        P[pv.off_ln_beta[l]:pv.off_ln_beta[l] + 128] = 0.1 * rs.standard_normal(128)
    w = P[pv.off_head:pv.off_head + 128 * pv.head_dim].reshape(128, -1)
    w[:, :-1] *= np.float32(head)
    model.set_params(P)
    model.collect()
    state, rng, done = gym.state(), gym.rng(), gym.done()
    last = model.download_slots()["obs"][T]
    tiles, tiles_head = collect_with_view(mg, gym, without_planes(model.policy()), T, last)
    mg.h2d(gym.buf.state, state)
    mg.h2d(gym.buf.rng, rng)
    mg.h2d(gym.buf.done, done)
    model.collect()
    return model, model.download_slots(), tiles, tiles_head


@pytest.mark.parametrize("env,n,tile,layers,scale", [
    ("cartpole", 64, 16, 2, 4),
    ("cartpole", 2048, 16, 3, 5),   # two workgroups' rotations of the weights
    ("cartpole", 8192, 32, 2, 4),
    ("cartpole", 32768, 64, 1, 1),
    ("cartpole", 32768, 64, 2, 4),
    ("voxelnav16", 8192, 32, 2, 4),
    ("voxelnav16", 32768, 64, 2, 4),
])
def test_row_heads(mg, env, n, tile, layers, scale):
    model, _, tiles, want = both(mg, env, n, 1, layers, scale, 1.0)
    pv = model.policy()
    obs, head = mg.DeviceBuffer.from_array(tiles["obs"][1]), mg.DeviceBuffer(want.nbytes)
    rc = ctypes.CDLL(LIB).mg_test_row_heads(ctypes.byref(pv), ctypes.c_void_p(obs.ptr), n, tile,
                                            ctypes.c_void_p(head.ptr))
    assert rc == 0, rc
    assert_bit_exact(head.download(np.float32, want.shape), want, f"{env} heads of {n} rows")


@pytest.mark.parametrize("env,n", [
    ("cartpole", 4096),      # 16-row tiles on pairs
    ("cartpole", 8192),
    ("cartpole", 16384),     # two shares
    ("cartpole", 32832),     # one
    ("voxelnav16", 16384),
    ("voxelnav16", 32832),
])
@pytest.mark.parametrize("head", [1.0, 16.0])
def test_actions(mg, env, n, head):
    """Heads of the initial size, and logits with a standard deviation of 1 to
    1.5: their edges are within the window (kLaneEdge)."""
    _, got, tiles, _ = both(mg, env, n, 64, 2, 4, head)
    for key in ("actions", "obs", "reward", "done"):
        assert_bit_exact(got[key], tiles[key], f"{env} {key}")


@pytest.mark.parametrize("n", [4096, 65536])
def test_actions_of_large_logits(mg, n):
    """A standard deviation of 20: the two logits differ by up to 1e-4, so an edge
    by up to a quarter of that. At most that share of the draws, times the two
    sides, is decided otherwise."""
    T = 32
    _, got, tiles, _ = both(mg, "cartpole", n, T, 2, 4, 256.0)
    differ = (got["actions"] != tiles["actions"]).any(0)
    assert differ.sum() <= max(1, n * T * 5e-5)
    for key in ("obs", "reward", "done"):
        assert_bit_exact(got[key][:, ~differ], tiles[key][:, ~differ], key)
