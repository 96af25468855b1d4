"""The forwards on binary16 pairs (policy_lane.h, policy_pair.h) at the edges of
their range:
partial last workgroups, shapes at the ends, and weights whose size would leave
binary16's range without the stored scales. Head values against a float64
network, collect teacher-forced against the oracle."""
import numpy as np
import pytest

from parity import ENVS, THREADS
from test_cpu_lane_limits import DEEPEST
from test_gpu_collect import run_collect_parity

pytestmark = pytest.mark.gpu


def network64(pv, P, obs):
    """model/ppo.h:575-626 in float64."""
    P = P.astype(np.float64)
    E, H, O, HD = 128, pv.hidden, pv.obs_dim, pv.head_dim

    def mat(off, r, c):
        return P[off:off + r * c].reshape(r, c)

    def ln(h, l):
        d = h - h.mean(1, keepdims=True)
        xn = d / np.sqrt((d * d).mean(1, keepdims=True) + 1e-5)
        return xn * P[pv.off_ln_gamma[l]:pv.off_ln_gamma[l] + E] + P[pv.off_ln_beta[l]:pv.off_ln_beta[l] + E]

    h = obs.astype(np.float64) @ mat(pv.off_in_w, O, E) + P[pv.off_in_b:pv.off_in_b + E]
    for l in range(pv.layers):
        h = h + np.maximum(ln(h, l) @ mat(pv.off_up[l], E, H), 0) @ mat(pv.off_down[l], H, E)
    return ln(h, pv.layers) @ mat(pv.off_head, E, HD)


@pytest.mark.parametrize("env,rows,layers,scale,how", [
    ("cartpole", 8193, 2, 4, "init"),          # the first row count of the path: one row in the last workgroup
    ("cartpole", 12288, 2, 4, "init"),
    ("cartpole", 128 * 97 + 33, 1, 1, "init"),  # a wave and a row; the least hidden width
    ("cartpole_continuous", 12300, 4, 8, "init"),
    ("voxelnav16", 12416, 2, 4, "init"),
    ("voxelnav", 12417, 8, 1, "init"),         # the deepest, 40 observation floats
    ("cartpole", 12300, 2, 4, "large"),        # up x 2^40, down x 2^-40, gamma x 300
    ("cartpole", 12300, 2, 4, "small"),        # up x 2^-30, gamma x 2^-12
    ("cartpole", 12300, 2, 4, "outlier"),      # one weight 2^12 times the others
    ("cartpole", 12300, 2, 4, "zero"),         # a block's matrices all zero
    ("cartpole", 12300, 2, 4, "far"),          # observations of 1e6
    # 16-row tiles on pairs (policy_pair.h)
    ("cartpole", 1, 2, 4, "init"),
    ("cartpole", 8192, 2, 4, "init"),
    ("voxelnav16", 17, 3, 3, "init"),          # groups of hidden units uneven over the waves
    ("voxelnav", 1000, 8, 8, "init"),          # the largest policy
    ("cartpole_continuous", 100, 1, 1, "init"),  # waves without a group
    ("cartpole", 1000, 2, 4, "large"),
    ("cartpole", 1000, 2, 4, "small"),
    ("cartpole", 1000, 2, 4, "outlier"),
    ("cartpole", 1000, 2, 4, "zero"),
    ("cartpole", 1000, 2, 4, "far"),
])
def test_forward_lane(mg, orc, env, rows, layers, scale, how):
    """As far from float64 as fp32 sums are on the same rows. The oracle adds a
    block's products before it adds them to the residual stream, once per block;
    the kernel, like the fp32 tiles, adds them onto the stream 16 at a time, up
    to 3 * 1024 / 16 = 192 roundings at the stream's size. The fp32 tiles are 0.9
    to 2.9 times as far as the oracle on these rows, this 0.9 to 2.5."""
    gym = mg.Gym(ENVS[env][1], 64, 0)
    model = mg.PPOModel(gym, horizon=1, layers=layers, scale=scale)
    pv, rs = model.pv, np.random.default_rng(5)
    P = model.params()
    EH = 128 * pv.hidden
    P[pv.off_in_b:pv.off_in_b + 128] = 0.1 * rs.standard_normal(128)
    for l in range(layers + 1):
        P[pv.off_ln_gamma[l]:pv.off_ln_gamma[l] + 128] = 1 + 0.1 * rs.standard_normal(128)
        P[pv.off_ln_beta[l]:pv.off_ln_beta[l] + 128] = 0.1 * rs.standard_normal(128)
    up, down = (slice(o[0], o[0] + EH) for o in (pv.off_up, pv.off_down))
    gamma = slice(pv.off_ln_gamma[0], pv.off_ln_gamma[0] + 128)
    if how == "large":
        P[up] *= np.float32(2.0 ** 40)
        P[down] *= np.float32(2.0 ** -40)
        P[gamma] *= 300
    elif how == "small":
        P[up] *= np.float32(2.0 ** -30)
        P[gamma] *= np.float32(2.0 ** -12)
    elif how == "outlier":
        P[pv.off_up[0] + 77] *= 4096
        P[pv.off_down[1] + 1234] *= 4096
    elif how == "zero":
        P[up] = 0
        P[down] = 0
    model.set_params(P)
    obs = (rs.standard_normal((rows, gym.obs_dim)) * (1e6 if how == "far" else 1.5)).astype(np.float32)
    want = network64(pv, P, obs)
    d = orc.dims(ENVS[env][0], hidden=pv.hidden, layers=layers)
    got, plain = (np.abs(x - want) for x in (model.forward(obs), orc.forward(d, P, obs, threads=THREADS)))
    print("times the oracle's error:", np.linalg.norm(got) / np.linalg.norm(plain), got.max() / plain.max())
    assert np.linalg.norm(got) <= 3 * np.linalg.norm(plain), (np.linalg.norm(got), np.linalg.norm(plain))
    assert got.max() <= 4 * plain.max(), (got.max(), plain.max())


@pytest.mark.parametrize("env,n,T,layers,scale,bf16", [
    ("cartpole", 8192, 2, 2, 4, False),              # the last env count of the 16-row tiles on pairs
    ("cartpole", 8192 + 64, 3, 2, 4, False),         # two shares of the hidden units
    ("cartpole", 16384, 2, 2, 4, False),
    ("cartpole_continuous", 10240, 2, 1, 1, False),  # two stages per share, one block
    ("voxelnav16", 8192, 2, 8, 1, False),            # a block too deep for the lane kernel's LDS: the 32-row tiles
    ("cartpole", 16384 + 64, 3, 2, 4, False),        # one share: half a workgroup at the end
    ("cartpole_continuous", 16448, 2, 1, 8, False),
    ("cartpole_continuous_clamp", 16384, 2, 8, 1, False),
    ("voxelnav16", 16448, 2, 2, 4, False),
    ("voxelnav", 32832, 2, 2, 4, False),
    ("cartpole", 16448, 2, 2, 4, True),
    ("voxelnav16", 32832, 2, 1, 2, True),
])
def test_collect_lane(mg, orc, env, n, T, layers, scale, bf16):
    import metalgym_amd

    orig = metalgym_amd.PPOModel

    class Model(orig):  # minibatches that divide the env count
        def __init__(self, gym, **kw):
            super().__init__(gym, minibatch=64, **kw)

    class Mg:
        Gym, PPOModel = mg.Gym, Model

    run_collect_parity(Mg, orc, env, n, T, layers=layers, scale=scale, bf16=bf16)


@pytest.mark.parametrize("env,shares,n,T,over", [
    ("cartpole", 2, 8256, 2, 0),
    ("voxelnav16", 2, 8192, 2, 0),   # W_in in LDS beside the deepest policy that leaves it room
    ("cartpole", 1, 16448, 2, 0),
    ("cartpole", 1, 16448, 2, 1),    # one block more: the tiles
    ("voxelnav16", 1, 16448, 1, 0),
    ("voxelnav16", 1, 16448, 1, 1),
])
def test_collect_lane_deepest(mg, orc, env, shares, n, T, over):
    """The deepest policy on the lane kernel and, over, the first past its LDS."""
    layers = DEEPEST[env, shares] + over
    assert 1 <= layers <= 8
    test_collect_lane(mg, orc, env, n, T, layers, 1, False)


@pytest.mark.parametrize("env,n,T,layers,scale", [
    # the tiles, where they fill the GPU evenly, and the lane kernels an env count on
    ("cartpole", 8192, 3, 1, 1),
    ("cartpole_continuous", 8192, 2, 1, 1),
    ("voxelnav16", 8192, 2, 2, 3),
    ("voxelnav16", 8256, 2, 2, 3),
    ("voxelnav16", 16320, 2, 1, 1),
    ("voxelnav16", 16384, 2, 1, 1),
    ("voxelnav", 32768, 1, 1, 1),
    ("voxelnav", 32832, 1, 1, 1),
])
def test_collect_small_networks(mg, orc, env, n, T, layers, scale):
    test_collect_lane(mg, orc, env, n, T, layers, scale, False)


@pytest.mark.parametrize("env,n0,n1,T", [
    ("voxelnav16", 8192, 16448, 32),   # two shares against one, both in the 32-row tiles' arithmetic
    ("cartpole", 8192, 16384, 96),     # 16-row tiles on pairs against two shares, the same
    ("cartpole", 12288, 16448, 96),    # two shares against one
])
def test_collects_take_the_same_actions(mg, env, n0, n1, T):
    """The first n0 of n1 envs and n0 envs alone start from the same seeds. Draws
    within rounding of a CDF edge are decided by the fp32 tiles' arithmetic in
    every kernel, so the rollouts must be the same step for step."""
    runs = []
    for n in (n0, n1):
        gym = mg.Gym(ENVS[env][1], n, 3)
        model = mg.PPOModel(gym, horizon=T, seed=3, minibatch=64)
        model.collect()
        runs.append(model.download_slots())
    small, large = runs
    for key in ("actions", "obs", "reward", "done"):
        assert np.array_equal(small[key], large[key][:, :n0]), f"{env} {key}"
    np.testing.assert_allclose(large["logp"][:, :n0], small["logp"], rtol=0, atol=1e-5)
