"""VoxelNav16's bit-grid rollout (rollout_voxelnav16.h) at its envs per wave and
odd forms, against the oracle: bit for bit, as tests/test_gpu_rollout.py."""
import numpy as np
import pytest

from parity import ENVS, THREADS, assert_bit_exact
from test_gpu_rollout import compare_gym

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,steps", [
    (1, 300),       # one env: the split kernel, as to 7
    (7, 70),
    (8, 70),
    (1027, 40),     # 8 envs per wave, the last partial (three of them)
    (9001, 12),     # 16 per wave, one in the last; rows that start off 16 bytes
    (32769, 5),     # 32 per wave, one in the last
])
def test_random(mg, orc, n, steps):
    eid, kernel = ENVS["voxelnav16"]
    gym, g = mg.Gym(kernel, n, 11), orc.GymState(eid, n, 11)
    for rep in range(2):
        bufs = gym.rollout_random(steps)
        acts, obs, rew, dn = gym.download_slots(bufs, steps)
        oa, oo, orw, od = orc.rollout(g, steps, random=True, threads=THREADS)
        for got, want, what in ((acts, oa, "actions"), (obs, oo, "obs"), (rew, orw, "reward"), (dn, od, "done")):
            assert_bit_exact(got, want, f"rep {rep} {what}")
        compare_gym(gym, g, f"rep {rep}")


def test_given_actions_and_a_callers_grid(mg, orc):
    """Actions outside 0 .. 5 (clamped by the env), and cells that are neither 0
    nor 1 (occupied where not 0), which an env that did not reset keeps."""
    eid, kernel = ENVS["voxelnav16"]
    n, steps = 70, 30
    gym, g = mg.Gym(kernel, n, 2), orc.GymState(eid, n, 2)
    gym.rollout_random(3)
    orc.rollout(g, 3, random=True, threads=THREADS)
    rs = np.random.default_rng(1)
    state = g.state.reshape(n, -1)
    grid = state[:, 32:]
    grid[grid != 0] = rs.choice(np.array([1, 2, 127, 128, 255], np.uint8), int((grid != 0).sum()))
    mg.h2d(gym.buf.state, state)
    actions = rs.integers(-2, 9, (steps, n)).astype(np.int32)
    _, obs, rew, dn = gym.rollout_given(steps, actions)
    _, oo, orw, od = orc.rollout(g, steps, random=False, actions_in=actions, threads=THREADS)
    assert_bit_exact(obs.download(np.float32, (steps, n, 30)), oo, "obs")
    assert_bit_exact(rew.download(np.float32, (steps, n)), orw, "reward")
    assert_bit_exact(dn.download(np.uint8, (steps, n)), od, "done")
    compare_gym(gym, g, "after")


def test_no_outputs(mg, orc):
    """Every slot output may be NULL: the state still advances alike."""
    eid, kernel = ENVS["voxelnav16"]
    gym, g = mg.Gym(kernel, 130, 3), orc.GymState(eid, 130, 3)
    mg._capi.check(mg.lib().mg_gym_rollout_random(gym.h, 9, None, None, None, None))
    orc.rollout(g, 9, random=True, threads=THREADS)
    compare_gym(gym, g, "no outputs")


def test_agents_outside_the_grid(mg, orc):
    """Positions that the caller wrote, on the grid's sides and far off them:
    every cell out there is occupied, and a step into the grid is allowed."""
    eid, kernel = ENVS["voxelnav16"]
    n, steps = 4096, 6
    gym, g = mg.Gym(kernel, n, 5), orc.GymState(eid, n, 5)
    gym.rollout_random(2)
    orc.rollout(g, 2, random=True, threads=THREADS)
    rs = np.random.default_rng(2)
    position = g.state.reshape(n, -1)[:, :12].view(np.int32)
    position[:] = np.where(rs.random((n, 3)) < 0.5, position,
                           rs.choice(np.array([-33, -3, -2, -1, 0, 15, 16, 17, 18, 31, 32, 48], np.int32), (n, 3)))
    mg.h2d(gym.buf.state, g.state)
    bufs = gym.rollout_random(steps)
    acts, obs, rew, dn = gym.download_slots(bufs, steps)
    oa, oo, orw, od = orc.rollout(g, steps, random=True, threads=THREADS)
    for got, want, what in ((acts, oa, "actions"), (obs, oo, "obs"), (rew, orw, "reward"), (dn, od, "done")):
        assert_bit_exact(got, want, what)
    compare_gym(gym, g, "after")


@pytest.mark.parametrize("n,lengths", [(131072, (1, 2)), (131073, (1, 2)), (196608, (4, 5))])
def test_few_steps_of_many_envs(mg, orc, n, lengths):
    """Either side of the split kernel's lines."""
    eid, kernel = ENVS["voxelnav16"]
    gym, g = mg.Gym(kernel, n, 3), orc.GymState(eid, n, 3)
    for steps in lengths:
        bufs = gym.rollout_random(steps)
        got = gym.download_slots(bufs, steps)
        want = orc.rollout(g, steps, random=True, threads=THREADS)
        for x, y, what in zip(got, want, ("actions", "obs", "reward", "done")):
            assert_bit_exact(x, y, f"{steps} steps {what}")
    compare_gym(gym, g, "after")
