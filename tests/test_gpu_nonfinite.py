"""Parameters that are not finite, in the kernels that split fp32 operands
(policy_lane.h, policy_pair.h): a head is finite exactly where the float64
network's is, with its relu (0 for NaN), and as close as elsewhere; a diverged
policy is not taken for a healthy one."""
import numpy as np
import pytest

from parity import ENVS

pytestmark = pytest.mark.gpu


def network64(pv, P, obs):
    """model/ppo.h:575-626 in float64, the relu 0 for NaN as in the kernels."""
    P = P.astype(np.float64)
    E, H, O, HD = 128, pv.hidden, pv.obs_dim, pv.head_dim

    def mat(off, r, c):
        return P[off:off + r * c].reshape(r, c)

    def ln(h, l):
        d = h - h.mean(1, keepdims=True)
        xn = d / np.sqrt((d * d).mean(1, keepdims=True) + 1e-5)
        return xn * mat(pv.off_ln_gamma[l], 1, E) + mat(pv.off_ln_beta[l], 1, E)

    h = obs.astype(np.float64) @ mat(pv.off_in_w, O, E) + mat(pv.off_in_b, 1, E)
    for l in range(pv.layers):
        v = ln(h, l) @ mat(pv.off_up[l], E, H)
        h = h + np.where(v > 0, v, 0) @ mat(pv.off_down[l], H, E)
    return ln(h, pv.layers) @ mat(pv.off_head, E, HD)


def spoil(pv, P, how):
    """Parameters P with one element changed."""
    P = P.copy()
    at, value = {
        "up inf": (pv.off_up[0] + 77, np.inf),
        "up -inf": (pv.off_up[1] + 78, -np.inf),
        "up nan": (pv.off_up[0] + 79, np.nan),
        "down inf": (pv.off_down[0] + 80, np.inf),
        "down nan": (pv.off_down[1] + 81, np.nan),
        "gamma inf": (pv.off_ln_gamma[0] + 7, np.inf),
        "gamma nan": (pv.off_ln_gamma[1] + 7, np.nan),
        "beta -inf": (pv.off_ln_beta[1] + 8, -np.inf),
        "final gamma inf": (pv.off_ln_gamma[2] + 9, np.inf),
    }[how]
    P[at] = value
    return P


def check_heads(pv, P, obs, got):
    with np.errstate(all="ignore"):
        want = network64(pv, P, obs)
    finite = np.isfinite(want).all(1)
    np.testing.assert_array_equal(np.isfinite(got).all(1), finite)
    assert not np.isfinite(got[~finite]).any(), "every column of such a row goes through the final LayerNorm"
    np.testing.assert_allclose(got[finite], want[finite], rtol=0, atol=1e-4)
    return finite


HOW = ["up inf", "up -inf", "up nan", "down inf", "down nan", "gamma inf", "gamma nan", "beta -inf", "final gamma inf"]


@pytest.mark.parametrize("how", HOW)
@pytest.mark.parametrize("rows", [1000, 8200])  # 16-row tiles on pairs, row per lane pair
def test_forward(mg, rows, how):
    gym = mg.Gym(ENVS["cartpole"][1], 64, 0)
    model = mg.PPOModel(gym, horizon=1)
    P = spoil(model.pv, model.params(), how)
    model.set_params(P)
    obs = np.random.default_rng(3).normal(0, 1.5, (rows, 4)).astype(np.float32)
    finite = check_heads(model.pv, P, obs, model.forward(obs))
    if how in ("up inf", "up -inf"):  # the unit is on in some rows and off in others
        assert 0.2 < finite.mean() < 0.8


@pytest.mark.parametrize("how", HOW)
@pytest.mark.parametrize("n", [64, 8256, 16448])  # 16-row tiles on pairs, two shares, one
def test_collect(mg, n, how):
    gym = mg.Gym(ENVS["cartpole"][1], n, 0)
    model = mg.PPOModel(gym, horizon=2, minibatch=64)
    P = spoil(model.pv, model.params(), how)
    model.set_params(P)
    model.collect()
    check_heads(model.pv, P, model.download_slots()["obs"][2], model.head())


@pytest.mark.parametrize("how", HOW)
def test_minibatch(mg, how):
    """The row pass computes the same heads, and a loss that is not finite
    reaches the gradient's norm."""
    n = 256
    gym = mg.Gym(ENVS["cartpole"][1], n, 0)
    model = mg.PPOModel(gym, horizon=2, minibatch=n)
    model.collect()
    P = spoil(model.pv, model.params(), how)
    model.set_params(P)
    model.train_block(1)
    finite = check_heads(model.pv, P, model.download_slots()["obs"][1], model.head())
    assert finite.all() or not np.isfinite(model.last_stats().grad_norm)
