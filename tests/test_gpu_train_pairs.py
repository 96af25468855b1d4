"""The fp32 PPO minibatch on binary16 pairs (policy_pair.h) and its weight
gradients on three bfloat16 planes, at the edges of their shapes: one minibatch
against the oracle's train step, and the operand copies that Adam keeps against
the parameters they stand for after many large steps."""
import numpy as np
import pytest

from parity import ENVS, check_minibatch
from test_gpu_lane import network64
from test_gpu_train import block_rows, setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("env,n,B,layers,scale", [
    ("cartpole", 64, 64, 1, 1),               # 4 groups of hidden units for 8 waves; 4 steps for 8 waves
    ("cartpole", 640, 320, 2, 3),             # 12 groups: waves of one and of two
    ("cartpole_continuous", 192, 192, 3, 5),  # 20 groups
    ("voxelnav16", 128, 128, 2, 2),           # one group per wave, 30 observation floats
    ("cartpole", 64, 64, 4, 8),               # gradient tiles that fill the GPU, fewer steps than waves
    ("cartpole_continuous", 320, 320, 4, 8),  # 20 steps of 16 rows over 8 waves
    ("cartpole", 4096, 4096, 4, 4),           # the first work of the row-split gradients
    ("cartpole", 128, 128, 5, 1),             # past the pair layout's LDS: the fp32 row pass
])
def test_minibatch(mg, orc, env, n, B, layers, scale):
    gym, model, d = setup(mg, orc, env, n, 2, B, layers=layers, scale=scale)
    s, p0 = model.download_slots(), model.params()
    model.train_block(1)
    check_minibatch(model, orc, d, orc.hparams(), p0, block_rows(s, n, B, 1), B)


@pytest.mark.parametrize("lr,epochs", [(3e-4, 2), (0.05, 5), (1.0, 3)])
def test_copies_follow_the_parameters(mg, lr, epochs):
    """Adam writes its planes with exponents made before the step, from the
    largest weight and from how far one step can move it. After training, the
    head that the next minibatch's row pass computes from them must be the
    parameters' (relative to the row's largest: 1e-4 as the policy heads
    elsewhere)."""
    n = 1024
    gym = mg.Gym(ENVS["cartpole"][1], n, 0)
    model = mg.PPOModel(gym, horizon=4, minibatch=256, lr=lr)
    model.collect()
    model.train(epochs)
    p, obs = model.params(), model.download_slots()["obs"]
    assert np.isfinite(p).all()
    model.train_block(5)  # slot 1, rows 256 .. 511
    want = network64(model.pv, p, obs[1][256:512])
    err = np.abs(model.head() - want) / np.maximum(1.0, np.abs(want).max(1, keepdims=True))
    assert float(err.max()) <= 1e-4, float(err.max())


@pytest.mark.parametrize("layers,lr", [(2, 3e-4), (2, 0.05), (2, 1.0), (5, 0.05)])
def test_copies_after_training(mg, layers, lr):
    """What a view hands out after training (exponents from the magnitudes that
    Adam keeps per tile) is what the same parameters give when they are set:
    every copy and the collects' exponents, bit for bit. 5 blocks: the fp32 row
    pass, whose Adam does not write the pair planes."""
    n = 512
    gym = mg.Gym(ENVS["cartpole"][1], n, 0)
    model = mg.PPOModel(gym, horizon=4, minibatch=256, layers=layers, lr=lr)
    count, halves = model.pv.count, 2 * model.pv.count

    def copies():
        pv = model.policy()
        scale = mg.d2h(pv.frag_fwd32_bf, np.uint16, (halves + 32,))[halves:].view(np.int32).reshape(2, 8)[:, :layers]
        cur = mg.d2h(pv.frag_fwd16_bf, np.uint16, (halves + 32,))[halves:].view(np.int32)[:2 * layers]
        got = {k: mg.d2h(getattr(pv, k), np.uint32, (count,)) for k in ("frag_fwd32", "frag_fwd16", "frag_bwd16")}
        got.update({k: mg.d2h(getattr(pv, k), np.uint16, (halves,)) for k in ("frag_fwd32_bf", "frag_fwd16_bf",
                                                                             "frag_bwd16_bf")})
        return dict(got, scale=scale, cur=cur)

    model.collect()
    for _ in range(3):
        model.train(2)
        got = copies()
        model.set_params(model.params())
        want = copies()
        for k in want:
            np.testing.assert_array_equal(got[k], want[k], err_msg=k)


@pytest.mark.parametrize("env,n,layers,scale", [
    ("cartpole_continuous", 16384, 4, 8),  # all rows in one workgroup: 128 steps a wave
    ("cartpole", 16384, 2, 4),             # row splits: 32, the most in one chain
    ("cartpole", 4160, 4, 8),              # 260 steps over 8 waves: chains that end short
    ("cartpole", 81920, 2, 4),             # row splits past it
    ("cartpole", 1088, 4, 8),              # 68 steps over 8 waves
])
def test_block_gradients_are_not_short(mg, env, n, layers, scale):
    """The block matrices' gradients against float64 sums of the captures they are
    made of: as close as fp32 sums, and not all a little too small, which the
    norm and the clip would pass on to every parameter. The first moment is
    fp32(1 - 0.9f) g clip; three roundings, the clip's two, common to all elements,
    are up to 1.2e-7 (2^-24 each) together."""
    gym = mg.Gym(ENVS[env][1], n, 0)
    model = mg.PPOModel(gym, horizon=1, minibatch=n, layers=layers, scale=scale)
    model.collect()
    model.train_block(0)
    pv, m = model.pv, model.adam_state()[0].astype(np.float64)
    norm = np.float32(model.last_stats().grad_norm)
    factor = float(np.float32(1) - np.float32(0.9)) * (float(np.float32(0.5) / (norm + np.float32(1e-6))) if norm > 0.5 else 1)
    x, v, dh, dv = (model.train_capture(k) for k in range(4))
    for l in (0, layers - 1):
        for off, a, b in ((pv.off_up[l], x[l], dv[l]), (pv.off_down[l], v[l], dh[l])):
            want = (a.astype(np.float64).T @ b.astype(np.float64)).ravel()
            got = m[off:off + want.size] / factor
            short = float(got @ want / (want @ want) - 1)
            err = float(np.linalg.norm(got - want) / np.linalg.norm(want))
            print(f"layer {l}: short by {short:.2e}, error {err:.2e}")
            assert abs(short) <= 2e-7 and err <= 4e-7
