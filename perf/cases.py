"""The work that a user of metalgym_amd has it do, as cases that can be timed and compared.

Every case goes through the package's public entry points (``Gym``, ``PPOModel`` and, where the
caller's data is already on the GPU, the C ABI behind them) and returns the whole of what the call
computes as views of the device buffers that the call wrote. Kinds:

* ``step``     one env step from the gym's action buffer: the smallest call there is.
* ``rollout``  a random-policy rollout of ``steps`` steps in one launch (no network).
* ``collect``  the whole rollout of a PPO iteration: policy forward, sampling, env step, GAE.
* ``forward``  the policy on given observation rows (acting, evaluation): any row count.
* ``train``    one epoch over a collected rollout, one Adam step per minibatch.

``exact`` repeats a CartPole family case in float64 with plain torch: generator, dynamics, network,
sampling, GAE, loss, gradients (autograd) and Adam. The voxel env has no such restatement here.
"""
import ctypes
import math

import numpy as np
import torch
import torch.nn.functional as F

import metalgym_amd as mg

ENVS = {  # kernel, observation floats, actions, float actions
    "cartpole": ("rollout_cartpole", 4, 2, False),
    "continuous": ("rollout_cartpole_continuous", 4, 1, True),
    "voxelnav16": ("rollout_voxelnav16", 30, 6, False),
}
EMBED = 128
LR = 3e-4
MOST_STEPS = 1 << 21  # env steps of the largest collect


def listed():
    return [
        # a caller that steps a handful of envs by hand: launch latency is the whole cost
        {"name": "step_64", "kind": "step", "env": "cartpole", "n": 64},
        # the README's env-only throughput run at its size, and at the size that fills the GPU
        {"name": "rollout_4096", "kind": "rollout", "env": "cartpole", "n": 4096, "steps": 32},
        {"name": "rollout_262144", "kind": "rollout", "env": "cartpole", "n": 262144, "steps": 32},
        # the same for an env whose state is a voxel grid of 4 KB
        {"name": "rollout_voxel_65536", "kind": "rollout", "env": "voxelnav16", "n": 65536, "steps": 32},
        # the collect of a PPO iteration: the README's 4096 envs, a large run, and as many envs as
        # the largest configuration has, with the voxel env between them
        {"name": "collect_4096", "kind": "collect", "env": "cartpole", "n": 4096, "steps": 32, "layers": 2, "scale": 4},
        {"name": "collect_65536", "kind": "collect", "env": "cartpole", "n": 65536, "steps": 32, "layers": 2, "scale": 4},
        {"name": "collect_262144", "kind": "collect", "env": "cartpole", "n": 262144, "steps": 8, "layers": 2, "scale": 4},
        {"name": "collect_voxel_16384", "kind": "collect", "env": "voxelnav16", "n": 16384, "steps": 16, "layers": 2,
         "scale": 4},
        # evaluation of a trained policy on recorded observations, an odd number of them, with bf16 matmuls
        {"name": "forward_bf16_100003", "kind": "forward", "env": "cartpole", "rows": 100003, "layers": 2, "scale": 4,
         "precision": "bf16"},
        # one epoch of PPO updates: the default policy and minibatch in both precisions, and a
        # deeper and wider Gaussian policy on large minibatches
        {"name": "train_4096", "kind": "train", "env": "cartpole", "n": 4096, "steps": 8, "minibatch": 4096, "layers": 2,
         "scale": 4, "precision": "fp32"},
        {"name": "train_bf16_4096", "kind": "train", "env": "cartpole", "n": 4096, "steps": 8, "minibatch": 4096,
         "layers": 2, "scale": 4, "precision": "bf16"},
        {"name": "train_wide_16384", "kind": "train", "env": "continuous", "n": 16384, "steps": 4, "minibatch": 16384,
         "layers": 4, "scale": 8, "precision": "fp32"},
    ]


def _spread(rng, lo, hi):
    """A whole number of [lo, hi], even over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["step", "rollout", "collect", "collect", "collect", "forward", "train", "train", "train"])
    if kind == "step":
        return {"kind": kind, "env": rng.choice(["cartpole", "continuous"]), "n": _spread(rng, 1, 65536)}
    if kind == "rollout":
        env = rng.choice(["cartpole", "continuous", "voxelnav16"])
        return {"kind": kind, "env": env, "n": _spread(rng, 64, 65536 if env == "voxelnav16" else 262144),
                "steps": rng.randint(1, 32)}
    layers, scale = rng.choice([1, 2, 2, 2, 3, 4]), rng.choice([1, 2, 4, 4, 4, 8])
    if kind == "collect":
        env = rng.choice(["cartpole", "cartpole", "continuous", "voxelnav16"])
        n = 64 * _spread(rng, 1, 4096 if env != "voxelnav16" else 256)
        n = n if n <= 4096 else n // 1024 * 1024
        if layers * scale > 8:  # no costlier than the default policy
            layers, scale = 2, 4
        return {"kind": kind, "env": env, "n": n, "steps": rng.randint(1, max(1, min(32, MOST_STEPS // n))),
                "minibatch": min(n, 1024) if n % 1024 == 0 else n, "layers": layers, "scale": scale}
    precision = rng.choice(["fp32", "fp32", "bf16"])
    if kind == "forward":
        return {"kind": kind, "env": rng.choice(["cartpole", "voxelnav16"]), "rows": _spread(rng, 1, 262144),
                "layers": layers, "scale": scale, "precision": precision}
    minibatch = 64 * _spread(rng, 1, 256)
    n = minibatch * rng.choice([1, 1, 2])
    if layers * scale > 16:
        layers, scale = 4, 4
    return {"kind": kind, "env": rng.choice(["cartpole", "continuous"]), "n": n, "steps": rng.randint(1, 4),
            "minibatch": minibatch, "layers": layers, "scale": scale, "precision": precision}


# ---- what a program holds before the call -------------------------------------------------------

_TYPES = {"f": "<f4", "i": "<i4", "b": "|u1"}


class _Device:
    """Device memory of the library as something torch can wrap without a copy. The tensor keeps
    this object, and this object the owner of the memory."""

    def __init__(self, owner, ptr, shape, kind):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (int(ptr), False), "shape": tuple(shape), "typestr": _TYPES[kind],
                                         "strides": None, "version": 2}


def _view(owner, ptr, shape, kind):
    return torch.as_tensor(_Device(owner, ptr, shape, kind), device="cuda")


def _weights(case, seed):
    """The policy's tensors in float32: the library's initial distributions (uniform, the same
    standard deviations), with the LayerNorm parameters moved off 1 and 0 as training does."""
    _, obs, act, cont = ENVS[case["env"]]
    L, H = case["layers"], EMBED * case["scale"]
    r = np.random.RandomState(seed % (1 << 32))

    def uniform(rows, cols, bound):
        return r.uniform(-bound, bound, (rows, cols)).astype(np.float32)

    w = {"in_w": uniform(obs, EMBED, math.sqrt(3 / obs)), "in_b": r.normal(0, 0.02, EMBED).astype(np.float32)}
    for l in range(L + 1):
        w["g%d" % l] = r.normal(1, 0.05, EMBED).astype(np.float32)
        w["b%d" % l] = r.normal(0, 0.02, EMBED).astype(np.float32)
    if cont:
        w["log_std"] = r.normal(-0.5, 0.1, act).astype(np.float32)
    for l in range(L):
        w["up%d" % l] = uniform(EMBED, H, math.sqrt(6 / EMBED))
        w["down%d" % l] = uniform(H, EMBED, math.sqrt(3 / H) / math.sqrt(L))
    w["head"] = np.concatenate([uniform(EMBED, act, 0.01 * math.sqrt(3)), uniform(EMBED, 1, math.sqrt(3 / EMBED))], 1)
    return w


def _offsets(case, pv):
    at = {"in_w": pv.off_in_w, "in_b": pv.off_in_b, "head": pv.off_head}
    for l in range(case["layers"] + 1):
        at["g%d" % l], at["b%d" % l] = pv.off_ln_gamma[l], pv.off_ln_beta[l]
    for l in range(case["layers"]):
        at["up%d" % l], at["down%d" % l] = pv.off_up[l], pv.off_down[l]
    if ENVS[case["env"]][3]:
        at["log_std"] = pv.off_log_std
    return at


def _gym_seed(seed):
    return seed % 1000003


def _model(case, seed, n, steps, minibatch=0):
    gym = mg.Gym(ENVS[case["env"]][0], n, _gym_seed(seed))
    model = mg.PPOModel(gym, scale=case["scale"], layers=case["layers"], lr=LR, horizon=steps, seed=_gym_seed(seed),
                        minibatch=minibatch, precision=case.get("precision", "fp32"))
    flat = np.zeros(model.pv.count, np.float32)
    at = _offsets(case, model.pv)
    for k, v in _weights(case, seed).items():
        flat[at[k]:at[k] + v.size] = v.ravel()
    model.set_params(flat)
    return gym, model


def _observations(case, seed, rows):
    """Observation rows as a rollout meets them: a CartPole's position, angle and their rates
    inside the termination bounds; a voxel env's cells in {0, 1} beside offsets in [-1, 1]."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    obs = ENVS[case["env"]][1]
    if case["env"] == "voxelnav16":
        x = (torch.rand(rows, obs, generator=g, device="cuda") < 0.25).float()
        x[:, -3:] = torch.rand(rows, 3, generator=g, device="cuda") * 2 - 1
        return x.contiguous()
    scale = torch.tensor([0.8, 0.7, 0.08, 0.9], device="cuda")
    return (torch.randn(rows, obs, generator=g, device="cuda") * scale).contiguous()


def _actions(case, seed):
    _, _, act, cont = ENVS[case["env"]]
    r = np.random.RandomState(seed % (1 << 32))
    return r.normal(0, 1, (case["n"], act)).astype(np.float32) if cont else r.randint(0, act, case["n"]).astype(np.int32)


def prepare(case, seed):
    _, obs, act, cont = ENVS[case["env"]]
    s = {"kind": case["kind"]}
    if case["kind"] in ("step", "rollout"):
        n = case["n"]
        s["gym"] = gym = mg.Gym(ENVS[case["env"]][0], n, _gym_seed(seed))
        s["out"] = {"rng": _view(gym, gym.buf.rng, (n,), "i"), "done": _view(gym, gym.buf.done, (n,), "b")}
        if case["kind"] == "step":
            gym.set_actions(_actions(case, seed))
            s["out"].update(obs=_view(gym, gym.buf.obs, (n, obs), "f"), reward=_view(gym, gym.buf.reward, (n,), "f"))
        else:
            T = s["steps"] = case["steps"]
            s["bufs"] = b = gym._slot_bufs(T)
            s["out"].update(actions=_view(b, b[0].ptr, (T, n, act) if cont else (T, n), "f" if cont else "i"),
                            obs=_view(b, b[1].ptr, (T, n, obs), "f"), reward=_view(b, b[2].ptr, (T, n), "f"),
                            dones=_view(b, b[3].ptr, (T, n), "b"))
        return s
    if case["kind"] == "forward":
        # a model of few envs, as a program that only acts has; the rows go through its head buffer
        s["gym"], s["model"] = _model(case, seed, 64, 1)
        s["obs"], s["rows"] = _observations(case, seed, case["rows"]), case["rows"]
        torch.cuda.synchronize()
        run(s)  # the head buffer grows to the row count on the first call
        return s
    n, T = case["n"], case["steps"]
    s["gym"], s["model"] = gym, m = _model(case, seed, n, T, case.get("minibatch", 0))
    sl = m.slots
    if case["kind"] == "collect":
        s["out"] = {"obs": _view(m, sl.obs, (T + 1, n, obs), "f"), "logp": _view(m, sl.logp, (T, n), "f"),
                    "actions": _view(m, sl.actions, (T, n, act) if cont else (T, n), "f" if cont else "i"),
                    "value": _view(m, sl.value, (T, n), "f"), "reward": _view(m, sl.reward, (T, n), "f"),
                    "done": _view(m, sl.done, (T, n), "b"), "adv": _view(m, sl.advantage, (T, n), "f"),
                    "ret": _view(m, sl.ret, (T, n), "f"), "rng": _view(m, gym.buf.rng, (n,), "i")}
        p, rows, hd = ctypes.c_void_p(), ctypes.c_uint32(), ctypes.c_uint32()
        mg._capi.check(mg.lib().mg_ppo_head(m.h, ctypes.byref(p), ctypes.byref(rows), ctypes.byref(hd)))
        s["out"]["head"] = _view(m, p.value, (n, act + 1), "f")
        return s
    m.collect()
    am, av, step = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_uint32()
    mg._capi.check(mg.lib().mg_ppo_adam_state(m.h, ctypes.byref(am), ctypes.byref(av), ctypes.byref(step)))
    count = (m.pv.count,)
    s["out"] = {"params": _view(m, m.pv.params, count, "f"), "m": _view(m, am.value, count, "f"),
                "v": _view(m, av.value, count, "f")}
    return s


def run(s):
    kind = s["kind"]
    if kind == "step":
        s["gym"].run()
        return s["out"]
    if kind == "rollout":
        s["gym"].rollout_random(s["steps"], s["bufs"])
        return s["out"]
    model = s["model"]
    if kind == "collect":
        model.collect()
        return s["out"]
    if kind == "train":
        model.train(1)
        return dict(s["out"], stats=model.train_stats())
    lib, rows = mg.lib(), s["rows"]
    mg._capi.check(lib.mg_ppo_forward(model.h, s["obs"].data_ptr(), rows))
    p, r, hd = ctypes.c_void_p(), ctypes.c_uint32(), ctypes.c_uint32()
    mg._capi.check(lib.mg_ppo_head(model.h, ctypes.byref(p), ctypes.byref(r), ctypes.byref(hd)))
    if s.get("head_at") != p.value:
        s["head_at"], s["head"] = p.value, _view(model, p.value, (rows, hd.value), "f")
    return {"head": s["head"]}


# ---- what a pass cannot do without ----------------------------------------------------------------

_STATE = {"cartpole": 20, "continuous": 20, "voxelnav16": 4128}


def work(case):
    _, obs, act, cont = ENVS[case["env"]]
    abytes = 4 * act if cont else 4
    if case["kind"] in ("step", "rollout"):
        n, T = case["n"], case.get("steps", 1)
        state = 2 * 20 if _STATE[case["env"]] < 64 else _STATE[case["env"]] + 32  # a grid is read, not rewritten
        return {"bytes": n * (state + 10) + n * T * (4 * obs + abytes + 5), "flops": 0}
    L, H, HD = case["layers"], EMBED * case["scale"], act + 1
    macs = obs * EMBED + 2 * L * EMBED * H + EMBED * HD
    params = obs * EMBED + EMBED + 2 * EMBED * (L + 1) + 2 * L * EMBED * H + EMBED * HD + (act if cont else 0)
    if case["kind"] == "forward":
        return {"bytes": 4 * (case["rows"] * (obs + HD) + params), "flops": 2 * macs * case["rows"]}
    n, T = case["n"], case["steps"]
    if case["kind"] == "collect":
        slots = n * T * (4 * obs + abytes + 4 * 5 + 1) + n * 4 * (obs + HD)
        return {"bytes": slots + n * (2 * min(_STATE[case["env"]], 64) + 10) + 4 * params, "flops": 2 * macs * n * (T + 1)}
    rows, steps = n * T, n * T // case["minibatch"]
    # forward, gradients of the activations (not of the observations) and of the weights; Adam
    # reads and writes parameters and both moments
    flops = rows * 2 * (3 * macs - obs * EMBED)
    return {"bytes": rows * (4 * obs + abytes + 12) + steps * 24 * params, "flops": flops}


def tolerance(case):
    kind = case["kind"]
    bf16 = case.get("precision") == "bf16"
    if kind in ("step", "rollout"):
        return {"rel": 1e-6, "max": 1e-5, "differ": 0.0}
    if kind == "forward":
        return {"rel": 1e-2, "max": 0.1} if bf16 else {"rel": 1e-5, "max": 2e-4}
    if kind == "collect":
        # whole rollouts: an action may differ where its draw falls on the edge of the policy's CDF
        return {"rel": 5e-6, "max": 5e-4, "differ": 1e-4}
    # a hidden unit within rounding of 0 may be on in one implementation and off in another, which
    # moves one of its minibatch * units * layers shares of the gradients; without one, 4e-5 off
    # float64 on the default policy
    one = (case["minibatch"] * EMBED * case["scale"] * case["layers"]) ** -0.5
    return {"rel": 2e-2, "max": 0.9} if bf16 else {"rel": 2e-4 + 2 * one, "max": 0.5}


# ---- the same in float64, with plain torch --------------------------------------------------------

_M32 = 0xFFFFFFFF


class _Rng:
    """One xorshift32 stream per env (shifts 13, 17, 5) in int64."""

    def __init__(self, n, seed):
        i = torch.arange(n, dtype=torch.int64, device="cuda")
        s = ((i * 2654435761 + 1) & _M32) ^ ((seed * 0x9E3779B9) & _M32)
        self.s = torch.where(s == 0, torch.full_like(s, 0x6D2B79F5), s)

    def next(self, where=None):
        s = self.s
        s = s ^ ((s << 13) & _M32)
        s = s ^ (s >> 17)
        s = s ^ ((s << 5) & _M32)
        self.s = s if where is None else torch.where(where, s, self.s)
        return s

    def uniform(self, lo=0.0, hi=1.0, where=None):
        return lo + (hi - lo) * ((self.next(where) >> 8).double() / 16777216.0)

    def int32(self):
        return torch.where(self.s >= 1 << 31, self.s - (1 << 32), self.s).int()


class _Pole:
    """CartPole (Barto, Sutton and Anderson 1983), with integer or float actions."""

    def __init__(self, n, seed, cont):
        self.rng, self.cont = _Rng(n, seed), cont
        self.s = torch.zeros(n, 4, dtype=torch.float64, device="cuda")
        self.steps = torch.zeros(n, dtype=torch.int64, device="cuda")
        self.done = torch.ones(n, dtype=torch.bool, device="cuda")

    def step(self, action):
        d = self.done
        fresh = torch.stack([self.rng.uniform(-0.05, 0.05, d) for _ in range(4)], 1)
        self.s = torch.where(d[:, None], fresh, self.s)
        self.steps = torch.where(d, torch.zeros_like(self.steps), self.steps) + 1
        x, xd, th, thd = self.s.unbind(1)
        force = 10 * torch.tanh(action[:, 0]) if self.cont else torch.where(action == 1, 10.0, -10.0).double()
        sin, cos = torch.sin(th), torch.cos(th)
        temp = (force + 0.05 * thd * thd * sin) / 1.1
        tha = (9.8 * sin - cos * temp) / (0.5 * (4 / 3 - 0.1 * cos * cos / 1.1))
        xa = temp - 0.05 * tha * cos / 1.1
        self.s = torch.stack([x + 0.02 * xd, xd + 0.02 * xa, th + 0.02 * thd, thd + 0.02 * tha], 1)
        self.done = (self.s[:, 0].abs() > 2.4) | (self.s[:, 2].abs() > 12 * 2 * math.pi / 360) | (self.steps >= 500)
        return self.s


def _rounded(x, bf16):
    return x.float().bfloat16().double() if bf16 else x


def _network(t, x, layers, bf16=False):
    h = x @ t["in_w"] + t["in_b"]
    for l in range(layers):
        y = F.layer_norm(h, (EMBED,), t["g%d" % l], t["b%d" % l], eps=1e-5)
        v = torch.relu(_rounded(y, bf16) @ _rounded(t["up%d" % l], bf16))
        h = h + _rounded(v, bf16) @ _rounded(t["down%d" % l], bf16)
    return F.layer_norm(h, (EMBED,), t["g%d" % layers], t["b%d" % layers], eps=1e-5) @ t["head"]


def _tensors(case, seed):
    return {k: torch.tensor(v, dtype=torch.float64, device="cuda") for k, v in _weights(case, seed).items()}


def _sample(t, head, act, cont, rng):
    if cont:
        u1 = 1 - rng.uniform()
        u2 = rng.uniform()
        z = (torch.sqrt(-2 * torch.log(u1)) * torch.cos(2 * math.pi * u2))[:, None]
        a = head[:, :act] + torch.exp(t["log_std"]) * z
        return a, (-0.5 * z * z - t["log_std"] - 0.5 * math.log(2 * math.pi)).sum(1)
    lp = torch.log_softmax(head[:, :act], 1)
    u = rng.uniform()
    a = (u[:, None] >= torch.cumsum(torch.exp(lp), 1)[:, :-1]).sum(1)
    return a, lp.gather(1, a[:, None])[:, 0]


def _collected(case, seed):
    _, _, act, cont = ENVS[case["env"]]
    n, T, L = case["n"], case["steps"], case["layers"]
    t, env = _tensors(case, seed), _Pole(n, _gym_seed(seed), cont)
    zero = torch.zeros(n, act, dtype=torch.float64, device="cuda") if cont else torch.zeros(n, dtype=torch.int64,
                                                                                         device="cuda")
    obs = [env.step(zero)]  # the first collect takes one step with action 0
    got = {k: [] for k in ("actions", "logp", "value", "done")}
    for _ in range(T):
        head = _network(t, obs[-1], L)
        a, lp = _sample(t, head, act, cont, env.rng)
        obs.append(env.step(a))
        for k, v in (("actions", a), ("logp", lp), ("value", head[:, act]), ("done", env.done)):
            got[k].append(v)
    out = {k: torch.stack(v) for k, v in got.items()}
    out["obs"], out["head"] = torch.stack(obs), _network(t, obs[-1], L)
    out["reward"] = torch.ones(T, n, dtype=torch.float64, device="cuda")
    adv, nxt, last = [], out["head"][:, act], torch.zeros(n, dtype=torch.float64, device="cuda")
    for k in reversed(range(T)):
        live = 1.0 - out["done"][k].double()
        last = out["reward"][k] + 0.99 * nxt * live - out["value"][k] + 0.99 * 0.95 * live * last
        nxt = out["value"][k]
        adv.insert(0, last)
    out["adv"] = torch.stack(adv)
    out["ret"] = out["adv"] + out["value"]
    if not cont:
        out["actions"] = out["actions"].int()
    out["done"], out["rng"] = out["done"].to(torch.uint8), env.rng.int32()
    return out


def _order(seed, blocks):
    """The minibatch order of the first epoch: Fisher-Yates with SplitMix64."""
    s, mask = 0x4D47534855460000 ^ seed, (1 << 64) - 1
    order = list(range(blocks))
    for i in range(blocks, 1, -1):
        s = (s + 0x9E3779B97F4A7C15) & mask
        z = ((s ^ (s >> 30)) * 0xBF58476D1CE4E5B9) & mask
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
        j = (z ^ (z >> 31)) % i
        order[i - 1], order[j] = order[j], order[i - 1]
    return order


def _trained(case, seed):
    _, obs, act, cont = ENVS[case["env"]]
    c = _collected(dict(case, precision="fp32"), seed)
    n, B, L, bf16 = case["n"], case["minibatch"], case["layers"], case["precision"] == "bf16"
    t = _tensors(case, seed)
    m, v = ({k: torch.zeros_like(x) for k, x in t.items()} for _ in range(2))
    rows, stats, step = [], [], 0
    for block in _order(_gym_seed(seed), case["steps"] * (n // B)):
        at = (block // (n // B), slice(block % (n // B) * B, block % (n // B) * B + B))
        for x in t.values():
            x.requires_grad_(True)
        head = _network(t, c["obs"][at], L, bf16)
        adv, a = c["adv"][at], c["actions"][at]
        adv = (adv - adv.mean()) / (adv.std(unbiased=False) + 1e-8)
        if cont:
            ls = t["log_std"]
            lp = (-0.5 * ((a - head[:, :act]) * torch.exp(-ls)) ** 2 - ls - 0.5 * math.log(2 * math.pi)).sum(1)
            entropy = (ls + 0.5 * math.log(2 * math.pi) + 0.5).sum().expand(B)
        else:
            every = torch.log_softmax(head[:, :act], 1)
            lp, entropy = every.gather(1, a.long()[:, None])[:, 0], -(torch.exp(every) * every).sum(1)
        ratio = torch.exp(lp - c["logp"][at])
        policy = -torch.minimum(ratio * adv, torch.clamp(ratio, 0.8, 1.2) * adv)
        value = 0.5 * 0.5 * (head[:, act] - c["ret"][at]) ** 2
        (policy + value - 0.01 * entropy).mean().backward()
        step += 1
        with torch.no_grad():
            norm = torch.sqrt(sum((x.grad ** 2).sum() for x in t.values()))
            clip = torch.where(norm > 0.5, 0.5 / (norm + 1e-6), torch.ones_like(norm))
            for k, x in t.items():
                g = x.grad * clip
                m[k] = 0.9 * m[k] + 0.1 * g
                v[k] = 0.999 * v[k] + 0.001 * g * g
                t[k] = (x - LR * (m[k] / (1 - 0.9 ** step)) / (torch.sqrt(v[k] / (1 - 0.999 ** step)) + 1e-8)).detach()
            stats.append(torch.stack([policy.mean(), value.mean(), entropy.mean(), (c["logp"][at] - lp).mean(),
                                      ((ratio - 1).abs() > 0.2).double().mean(), norm]))
    # the arena: vectors first, then the matrices, each padded to a multiple of 128 elements
    names = ["in_w", "in_b"] + [k + str(l) for l in range(L + 1) for k in "gb"] + (["log_std"] if cont else [])
    names += [k + str(l) for l in range(L) for k in ("up", "down")] + ["head"]

    def arena(parts):
        return torch.cat([F.pad(parts[k].detach().reshape(-1), (0, -parts[k].numel() % 128)) for k in names])

    return {"params": arena(t), "m": arena(m), "v": arena(v), "stats": torch.stack(stats)}


def exact(case, seed):
    kind = case["kind"]
    _, _, act, cont = ENVS[case["env"]]
    if kind == "forward":
        with torch.no_grad():
            return {"head": _network(_tensors(case, seed), _observations(case, seed, case["rows"]).double(),
                                     case["layers"], case["precision"] == "bf16")}
    if not case["env"] in ("cartpole", "continuous"):
        return None  # the grid env's rollouts have no short restatement
    if kind == "collect":
        with torch.no_grad():
            return _collected(case, seed)
    if kind == "train":
        # bf16 gradients: the rounding of the backward's operands is not restated
        return None if case["precision"] == "bf16" else _trained(case, seed)
    n, T = case["n"], case.get("steps", 1)
    env, actions, obs, dones = _Pole(n, _gym_seed(seed), cont), [], [], []
    for _ in range(T):
        if kind == "step":
            a = torch.as_tensor(_actions(case, seed), device="cuda")
            a = a.double() if cont else a
        else:
            a = env.rng.uniform(-1.0, 1.0)[:, None] if cont else env.rng.next() % act
        obs.append(env.step(a))
        actions.append(a if cont else a.int())
        dones.append(env.done.to(torch.uint8))
    out = {"rng": env.rng.int32(), "done": dones[-1]}
    if kind == "step":
        return dict(out, obs=obs[0], reward=torch.ones(n, dtype=torch.float64, device="cuda"))
    return dict(out, actions=torch.stack(actions), obs=torch.stack(obs), dones=torch.stack(dones),
                reward=torch.ones(T, n, dtype=torch.float64, device="cuda"))
