"""Parameters that are not finite, or near the end of fp32's range, in the kernels that split fp32 operands
(policy_lane.h, policy_pair.h): a head is finite exactly where the float64
network's is, with its relu (0 for NaN), and as close as elsewhere; a diverged
policy is not taken for a healthy one."""
import numpy as np
import pytest

from parity import ENVS

pytestmark = pytest.mark.gpu


def network(pv, P, obs, dtype):
    """model/ppo.h:575-626 in dtype, the relu 0 for NaN as in the kernels."""
    P = P.astype(dtype)
    E, H, O, HD = 128, pv.hidden, pv.obs_dim, pv.head_dim

    def mat(off, r, c):
        return P[off:off + r * c].reshape(r, c)

    def ln(h, l):
        d = h - h.mean(1, keepdims=True)
        xn = d * (1 / np.sqrt((d * d).mean(1, keepdims=True) + dtype(1e-5)))
        return xn * mat(pv.off_ln_gamma[l], 1, E) + mat(pv.off_ln_beta[l], 1, E)

    h = obs.astype(dtype) @ mat(pv.off_in_w, O, E) + mat(pv.off_in_b, 1, E)
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
        want = network(pv, P, obs, np.float64)
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


def shifted(pv, P):
    """P with betas, which rows too long for fp32's squares come down to."""
    P = P.copy()
    for l in range(pv.layers + 1):
        P[pv.off_ln_beta[l]:pv.off_ln_beta[l] + 128] = np.random.default_rng(l).normal(0, 0.5, 128)
    return P


@pytest.mark.parametrize("rows", [1000, 8200])
def test_forward_of_huge_rows(mg, rows):
    """Observations to 1e35: past about 1e19 the squares of a row's deviations
    overflow, LayerNorm divides by infinity and leaves beta."""
    gym = mg.Gym(ENVS["cartpole"][1], 64, 0)
    model = mg.PPOModel(gym, horizon=1)
    P = shifted(model.pv, model.params())
    model.set_params(P)
    obs = np.random.default_rng(3).normal(0, 1.5, (rows, 4)).astype(np.float32)
    obs *= np.float32(10.0) ** np.array([0, 10, 17, 21, 25, 30, 35], np.float32)[np.arange(rows) % 7, None]
    with np.errstate(over="ignore"):
        want = network(model.pv, P, obs, np.float32)
    np.testing.assert_allclose(model.forward(obs), want, rtol=0, atol=1e-4)


@pytest.mark.parametrize("n", [64, 8256, 16448])
def test_collect_of_huge_rows(mg, n):
    gym = mg.Gym(ENVS["cartpole"][1], n, 0)
    model = mg.PPOModel(gym, horizon=2, minibatch=64)
    pv = model.pv
    P = shifted(pv, model.params())
    P[pv.off_in_w:pv.off_in_w + 4 * 128] *= np.float32(1e33)
    model.set_params(P)
    model.collect()
    with np.errstate(over="ignore"):
        want = network(pv, P, model.download_slots()["obs"][2], np.float32)
    np.testing.assert_allclose(model.head(), want, rtol=0, atol=1e-4)


@pytest.mark.parametrize("rows", [1000, 8200])
def test_blocks_with_units_far_apart(mg, rows):
    """One up weight of 1e36: the first block's unit is 2^-100 of the second's."""
    gym = mg.Gym(ENVS["cartpole"][1], 64, 0)
    model = mg.PPOModel(gym, horizon=1)
    P = shifted(model.pv, model.params())
    P[model.pv.off_up[0] + 77] = 1e36
    model.set_params(P)
    obs = np.random.default_rng(3).normal(0, 1.5, (rows, 4)).astype(np.float32)
    with np.errstate(over="ignore"):
        want = network(model.pv, P, obs, np.float32)
    got = model.forward(obs)
    assert np.isfinite(got).all()
    # where the unit is on, the row is too long for fp32's squares
    pv = model.pv
    beta, head = P[pv.off_ln_beta[2]:pv.off_ln_beta[2] + 128], P[pv.off_head:pv.off_head + 384].reshape(128, 3)
    on = np.abs(want - beta @ head).max(1) < 1e-5
    assert 0.2 < on.mean() < 0.8
    np.testing.assert_allclose(got[on], want[on], rtol=0, atol=1e-4)
