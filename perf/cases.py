"""The work that a user of this package has it do, as measurable cases.

Learner updates (DQN, SAC, PPO, recurrent PPO) as their captured steps,
acting steps, single layers (a convolution, a linear layer, a GRU unroll)
forward and backward as captured train steps, and a prioritized replay draw; each
through the package's public entry points, with float32 weights and the
uint8 frames or float32 vectors those networks read.

`exact` computes the same outputs in float64 with torch alone.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch
import torch.nn.functional as F

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "tt-rl_amd"))

FRAME_SCALE = float(np.float32(1.0 / 255.0))
TOWER = ((32, 8, 4), (64, 4, 2), (64, 3, 1))  # out channels, kernel, stride
FRAMES = (36, 52, 68, 84, 100)  # sizes that every stage of the tower covers without a rest
B1, B2 = 0.9, 0.999
# The learning rates are those near the end of an anneal, and Adam's epsilon
# of the SAC and PPO cases is 1e-5.  At the start's rates a PPO pass of 16
# steps is no longer a function of its inputs to float32: a ReLU gate or a
# clip that rounding decides moves a gradient by 1e-3, and the steps after it
# multiply that (moments of two correct float32 orders 4e-2 apart).
DQN_LR, DQN_EPS, SAC_LR, PPO_LR, EPS = 1e-5, 1.5e-4, 1e-4, 5e-7, 1e-5


# ------------------------------------------------------------------ cases ---

def listed() -> list:
    return [
        # one environment acting greedily on stacked frames: the smallest call, launches and one wait
        {"name": "act_greedy_1", "kind": "act_greedy", "lanes": 1, "channels": 4, "frame": 84, "actions": 6},
        # a vector environment of 16 lanes sampling from the squashed Gaussian policy
        {"name": "act_squashed_16", "kind": "act_squashed", "lanes": 16, "obs": 11, "act": 3, "hidden": 256},
        # the Atari DQN update of the headline benchmark, batches resident in two input slots
        {"name": "dqn_32", "kind": "dqn", "batch": 32, "channels": 4, "frame": 84, "actions": 6, "double": True,
         "read": False},
        # a small-frame RGB task at a ragged batch, the metrics read back after every update
        {"name": "dqn_75_rgb52", "kind": "dqn", "batch": 75, "channels": 3, "frame": 52, "actions": 9,
         "double": False, "read": True},
        # the Hopper-shaped SAC update of the benchmark (the fused stages)
        {"name": "sac_256", "kind": "sac", "batch": 256, "obs": 11, "act": 3, "hidden": 256},
        # a larger robot, a ragged batch and wider networks (the per-layer path)
        {"name": "sac_500_wide", "kind": "sac", "batch": 500, "obs": 27, "act": 8, "hidden": 300},
        # one PPO update: 8 environments x 128 steps, 4 epochs x 4 minibatches of 256
        {"name": "ppo_256", "kind": "ppo", "envs": 8, "steps": 128, "minibatch": 256, "epochs": 4, "channels": 4,
         "frame": 84, "actions": 18},
        # one recurrent PPO update: 16 environments x 128 steps, sequences of 32 through a GRU of 512
        {"name": "rppo_512", "kind": "rppo", "envs": 16, "steps": 128, "minibatch": 512, "epochs": 4, "channels": 4,
         "frame": 84, "actions": 18, "hidden": 512, "seq": 32},
        # the encoder's second convolution alone, forward and both gradients, at a large batch
        {"name": "conv_1024", "kind": "conv", "batch": 1024, "channels": 32, "size": 20, "out": 64, "kernel": 4,
         "stride": 2, "frames": False},
        # a linear layer's forward and all its gradients at ragged rows and widths
        {"name": "linear_1000", "kind": "linear", "rows": 1000, "in": 777, "out": 500},
        # a recurrent memory at the package's default sizes, forward and backward through time
        {"name": "gru_16x24", "kind": "gru", "steps": 16, "batch": 24, "in": 512, "hidden": 128},
        # a prioritized batch drawn from a replay of stacked frames into a learner's buffers
        {"name": "replay_32", "kind": "replay", "batch": 32, "capacity": 16384, "lanes": 8, "n_step": 3,
         "frame": 84},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    kind = rng.choice(["act_greedy", "act_squashed", "dqn", "dqn", "sac", "sac", "ppo", "rppo", "conv", "conv",
                       "linear", "linear", "gru", "gru", "replay"])
    c = {"kind": kind}
    image = {"channels": rng.choice([1, 3, 4]), "frame": rng.choice(FRAMES)}
    vector = {"obs": rng.randint(3, 56), "act": rng.randint(1, 8), "hidden": rng.choice([64, 128, 200, 256, 300, 400])}
    if kind == "act_greedy":
        c.update(image, lanes=_log_int(rng, 1, 64), actions=rng.randint(2, 18))
    elif kind == "act_squashed":
        c.update(vector, lanes=_log_int(rng, 1, 128))
    elif kind == "dqn":
        c.update(image, batch=_log_int(rng, 16, 256), actions=rng.randint(2, 18), double=rng.random() < 0.5,
                 read=rng.random() < 0.5)
    elif kind == "sac":
        c.update(vector, batch=_log_int(rng, 32, 1024))
    elif kind == "ppo":
        envs, steps = rng.choice([4, 8, 16]), rng.choice([64, 100, 128])
        c.update(image, envs=envs, steps=steps, epochs=rng.randint(1, 2), actions=rng.randint(2, 18),
                 minibatch=_log_int(rng, max(32, envs * steps // 8), min(512, envs * steps // 2)))
        c["frame"] = rng.choice(FRAMES[:4])
    elif kind == "rppo":
        seq = rng.choice([8, 16, 32])
        envs, chunks = rng.choice([8, 12, 16]), rng.randint(1, 128 // seq)
        c.update(image, envs=envs, steps=seq * chunks, seq=seq, epochs=rng.randint(1, 2),
                 hidden=rng.choice([100, 128, 256, 512]), actions=rng.randint(2, 18))
        c["minibatch"] = seq * rng.randint(max(2, envs * chunks // 8), max(2, min(envs * chunks // 2, 512 // seq)))
        c["frame"] = rng.choice(FRAMES[:4])
    elif kind == "conv":
        if rng.random() < 0.3:  # a first layer: uint8 frames, no input gradient
            c.update(image, batch=_log_int(rng, 8, 512), out=rng.choice([16, 32]), kernel=8, stride=4, frames=True)
            c["size"] = c.pop("frame")
        else:
            kernel, stride = rng.choice([(4, 2), (3, 1), (5, 1), (2, 2)])
            c.update(batch=_log_int(rng, 8, 512), channels=rng.choice([16, 32, 48, 64]), out=rng.choice([20, 32, 64]),
                     kernel=kernel, stride=stride, size=kernel + stride * rng.randint(2, 8), frames=False)
    elif kind == "linear":
        c.update(rows=_log_int(rng, 16, 4096), out=_log_int(rng, 1, 1024))
        c["in"] = _log_int(rng, 4, 3136)
    elif kind == "gru":
        c.update(steps=_log_int(rng, 4, 64), batch=_log_int(rng, 1, 64), hidden=rng.choice([64, 100, 128, 250, 256, 512]))
        c["in"] = _log_int(rng, 32, 512)
    else:
        lanes = rng.choice([1, 4, 8])
        c.update(batch=_log_int(rng, 8, 512), capacity=lanes * _log_int(rng, 512, 2048), lanes=lanes,
                 n_step=rng.randint(1, 5), frame=rng.choice(FRAMES[:4]))
    return c


# ---------------------------------------------------- inputs and weights ----

def _sizes(frame: int) -> list:
    out = []
    for _, k, s in TOWER:
        frame = (frame - k) // s + 1
        out.append(frame)
    return out


def _tower_shapes(channels: int, frame: int) -> list:
    shapes, c = [], channels
    for o, k, _ in TOWER:
        shapes.append((o, c, k, k))
        c = o
    shapes.append((_sizes(frame)[-1] ** 2 * c, 512))
    return shapes


def _mlp_shapes(*widths) -> list:
    return list(zip(widths[:-1], widths[1:]))


def _weights(rng, shapes) -> list:
    """He-uniform weights (conv OIHW, linear (in, out)) each followed by its bias."""
    out = []
    for s in shapes:
        fan = int(np.prod(s[1:])) if len(s) == 4 else s[0]
        out.append(rng.uniform(-math.sqrt(6.0 / fan), math.sqrt(6.0 / fan), s).astype(np.float32))
        n = s[0] if len(s) == 4 else s[1]
        bias = (1, 1, 1, n) if len(s) == 4 else (1, n)
        out.append(rng.uniform(-1.0 / math.sqrt(fan), 1.0 / math.sqrt(fan), bias).astype(np.float32))
    return out


def _gru_weights(rng, features: int, hidden: int) -> list:
    bound = 1.0 / math.sqrt(hidden)
    return [rng.uniform(-bound, bound, s).astype(np.float32)
            for s in ((features, 3 * hidden), (hidden, 3 * hidden), (1, 3 * hidden), (1, 3 * hidden))]


def _dqn_data(case, seed):
    rng = np.random.default_rng(seed)
    B, A = case["batch"], case["actions"]
    shapes = _tower_shapes(case["channels"], case["frame"]) + [(512, A)]
    online, target = _weights(rng, shapes), _weights(rng, shapes)
    shape = (B, case["channels"], case["frame"], case["frame"])
    batches = [{"obs": rng.integers(0, 256, shape, dtype=np.uint8), "next_obs": rng.integers(0, 256, shape, dtype=np.uint8),
                "actions": rng.integers(0, A, B).astype(np.int64),
                "rewards": rng.choice(np.array([-1.0, 0.0, 1.0], np.float32), B, p=[0.05, 0.9, 0.05]),
                "dones": (rng.random(B) < 0.01).astype(np.float32), "discounts": np.full(B, 0.99 ** 3, np.float32),
                "is_weights": (1.0 - 0.6 * rng.random(B)).astype(np.float32)} for _ in range(2)]
    return online, target, batches


def _sac_data(case, seed):
    rng = np.random.default_rng(seed)
    B, O, A, H = case["batch"], case["obs"], case["act"], case["hidden"]
    policy = _weights(rng, _mlp_shapes(O, H, H) + [(H, A), (H, A)])
    critics = [_weights(rng, _mlp_shapes(O + A, H, H, 1)) for _ in range(2)]

    def normal(*s):
        return rng.standard_normal(s).astype(np.float32)

    batches = [{"obs": normal(B, O), "next_obs": normal(B, O), "actions": np.clip(normal(B, A), -1.0, 1.0),
                "rewards": normal(B), "dones": (rng.random(B) < 0.001).astype(np.float32),
                "discounts": np.full(B, 0.99, np.float32), "noise": normal(B, A), "next_noise": normal(B, A)}
               for _ in range(2)]
    return policy, critics, batches


def _rollout_data(case, seed):
    """Weights and one time-major rollout whose actions, log-probabilities
    and values come from the policy itself."""
    rng = np.random.default_rng(seed)
    T, N, A, H = case["steps"], case["envs"], case["actions"], case.get("hidden", 512)
    trunk = _weights(rng, _tower_shapes(case["channels"], case["frame"]))
    gru = _gru_weights(rng, 512, H) if "hidden" in case else []
    heads = _weights(rng, [(H, A), (H, 1)])
    frames = rng.integers(0, 256, (T, N, case["channels"], case["frame"], case["frame"]), dtype=np.uint8)
    dones = (rng.random((T, N)) < 0.01).astype(np.float32)
    r = {"obs": frames, "dones": dones,
         "rewards": rng.choice(np.array([-1.0, 0.0, 1.0], np.float32), (T, N), p=[0.05, 0.9, 0.05]),
         "last_values": rng.standard_normal(N).astype(np.float32)}
    p = [torch.from_numpy(w).cuda() for w in trunk + gru + heads]
    flat = frames.reshape((T * N,) + frames.shape[2:])
    feats = torch.cat([_encode(p[:8], torch.from_numpy(flat[i:i + 256]).cuda()) for i in range(0, T * N, 256)])
    if gru:
        L = case["seq"]
        r["hidden"] = (0.5 * rng.standard_normal((T // L, N, H))).astype(np.float32)
        r["starts"] = np.concatenate([(rng.random((1, N)) < 0.01).astype(np.float32), dones[:-1]])
        x = feats.reshape(T // L, L, N, 512).transpose(0, 1).reshape(L, -1, 512)
        starts = torch.from_numpy(r["starts"]).cuda().reshape(T // L, L, N).transpose(0, 1).reshape(L, -1, 1)
        h = _unroll(p[8:12], x, torch.from_numpy(r["hidden"]).cuda().reshape(-1, H), starts)
        feats = h.reshape(L, T // L, N, H).transpose(0, 1).reshape(T * N, H)
    logp = torch.log_softmax(feats @ p[-4] + p[-3], -1).cpu().numpy()
    r["values"] = (feats @ p[-2] + p[-1]).cpu().numpy().reshape(T, N)
    actions = np.argmax(logp + rng.gumbel(size=logp.shape), -1)
    r["actions"] = actions.reshape(T, N)
    r["logp"] = np.take_along_axis(logp, actions[:, None], -1).reshape(T, N)
    return trunk, gru, heads, r


def _conv_data(case, seed):
    rng = np.random.default_rng(seed)
    B, C, size = case["batch"], case["channels"], case["size"]
    weights = _weights(rng, [(case["out"], C, case["kernel"], case["kernel"])])
    if case["frames"]:
        x = rng.integers(0, 256, (B, C, size, size), dtype=np.uint8)
    else:  # NHWC, what a ReLU below hands over
        x = np.maximum(rng.standard_normal((B, size, size, C), dtype=np.float32), 0.0)
    side = (size - case["kernel"]) // case["stride"] + 1
    dy = rng.standard_normal((1, 1, B * side * side, case["out"]), dtype=np.float32)
    return weights, x, dy


def _linear_data(case, seed):
    rng = np.random.default_rng(seed)
    weights = _weights(rng, [(case["in"], case["out"])])
    return (weights, rng.standard_normal((case["rows"], case["in"])).astype(np.float32),
            rng.standard_normal((case["rows"], case["out"])).astype(np.float32))


def _gru_data(case, seed):
    rng = np.random.default_rng(seed)
    T, B, I, H = case["steps"], case["batch"], case["in"], case["hidden"]
    x = np.maximum(rng.standard_normal((T, B, I)), 0.0).astype(np.float32)  # what a ReLU trunk hands over
    return (_gru_weights(rng, I, H), x, (0.5 * rng.standard_normal((B, H))).astype(np.float32),
            (rng.random((T, B, 1)) < 0.02).astype(np.float32), rng.standard_normal((T, B, H)).astype(np.float32))


def _replay_data(case, seed):
    """A replay that has been filled to three quarters of its capacity."""
    rng = np.random.default_rng(seed)
    lanes = case["lanes"]
    steps = case["capacity"] // lanes * 3 // 4
    base = rng.integers(0, 256, (64, lanes, 4, case["frame"], case["frame"]), dtype=np.uint8)
    fields = {"actions": rng.integers(0, 6, (steps, lanes)), "rewards": rng.standard_normal((steps, lanes)).astype(np.float32),
              "ends": rng.random((steps, lanes)) < 0.004, "priorities": rng.exponential(1.0, (lanes, steps))}
    return base, fields, steps


# ----------------------------------------------------------- the package ----

def _device():
    from ttrl_amd.engine.device import open_device

    return open_device(0)


class _Memory:
    """A device array of the package, as torch sees foreign device memory."""

    def __init__(self, array):
        self.array = array
        self.__cuda_array_interface__ = {"shape": tuple(array.shape), "typestr": np.dtype(array.dtype).str,
                                         "data": (array.ptr, False), "version": 2, "strides": None}


def _see(x):
    return torch.as_tensor(_Memory(getattr(x, "data", x)), device="cuda")


def _load(module, arrays) -> None:
    module.load_state_dict(dict(zip(module.state_dict(), arrays)))


def _adam_state(optimizer) -> dict:
    return {"params": [_see(p) for p in optimizer.params], "m": [_see(m) for m in optimizer.m],
            "v": [_see(v) for v in optimizer.v]}


def _prepare_act_greedy(case, seed):
    from ttrl_amd.nets.acting import ActingNet, GreedyDecision
    from ttrl_amd.nets.build import build_q_net
    from ttrl_amd.spaces import ActionSpec, ObsSpec

    rng = np.random.default_rng(seed)
    n, shape = case["lanes"], (case["channels"], case["frame"], case["frame"])
    spec = ObsSpec.image(shape)
    net = build_q_net(spec, ActionSpec.discrete(case["actions"]), _device(), batch=n)
    _load(net, _weights(rng, _tower_shapes(*shape[:2]) + [(512, case["actions"])]))
    acting = ActingNet(net, spec, _device(), width=n, lanes=n, decision=GreedyDecision())
    obs = rng.integers(0, 256, (n,) + shape, dtype=np.uint8)
    acting.decide(np.zeros_like(obs))
    return {"run": lambda: acting.decide(obs)}


def _prepare_act_squashed(case, seed):
    from ttrl_amd.algos.gaussian import ActionScale
    from ttrl_amd.nets.acting import ActingNet, SquashedDecision
    from ttrl_amd.nets.build import build_sac_nets
    from ttrl_amd.spaces import ActionSpec, ObsSpec

    rng = np.random.default_rng(seed)
    n, O, A, H = case["lanes"], case["obs"], case["act"], case["hidden"]
    spec, act = ObsSpec.vector(O), ActionSpec.continuous(A)
    nets = build_sac_nets(spec, act, _device(), batch=n, critic_hidden=(H, H), encoder_kwargs={"hidden": (H, H)})
    _load(nets.policy, _weights(rng, _mlp_shapes(O, H, H) + [(H, A), (H, A)]))
    acting = ActingNet(nets.policy, spec, _device(), width=n, lanes=n,
                       decision=SquashedDecision(ActionScale(act, _device())))
    obs, noise = (rng.standard_normal((n, k)).astype(np.float32) for k in (O, A))
    acting.decide(np.zeros_like(obs), noise=noise)
    return {"run": lambda: acting.decide(obs, noise=noise)}


def _alternate(step, out):
    """Passes that take the two input slots in turn, the second one first:
    the update that captures the step has run on slot 0."""
    at = [0]

    def run():
        at[0] ^= 1
        got = step(at[0])
        return out if got is None else dict(out, metrics=got)

    return run


def _prepare_dqn(case, seed):
    from ttrl_amd.algos.dqn import DQNConfig, DQNLearner
    from ttrl_amd.spaces import ActionSpec, ObsSpec

    online, target, batches = _dqn_data(case, seed)
    cfg = DQNConfig(lr=DQN_LR, adam_eps=DQN_EPS, batch_size=case["batch"], double=case["double"], prioritized=True)
    learner = DQNLearner(ObsSpec.image((case["channels"], case["frame"], case["frame"])),
                         ActionSpec.discrete(case["actions"]), _device(), cfg=cfg, seed=0)
    _load(learner.online, online)
    _load(learner.target, target)
    step = learner.step
    step.enable_input_slots(2)
    for k in (1, 0):
        learner.load_batch(batches[k])
        step.flush_inputs()
        if k:
            step.slot_inputs(k)["_block"].copy_from(learner.inputs["_block"])
    learner.update()
    return {"learner": learner, "run": _alternate(step.run_slot if case["read"] else step.replay_slot,
                                                  _adam_state(learner.optimizer))}


def _prepare_sac(case, seed):
    from ttrl_amd.algos.sac import SACConfig, SACLearner
    from ttrl_amd.spaces import ActionSpec, ObsSpec

    policy, critics, batches = _sac_data(case, seed)
    H = case["hidden"]
    cfg = SACConfig(lr=SAC_LR, adam_eps=EPS, batch_size=case["batch"], critic_hidden=(H, H), policy_hidden=(H, H))
    learner = SACLearner(ObsSpec.vector(case["obs"]), ActionSpec.continuous(case["act"]), _device(), cfg=cfg, seed=0)
    _load(learner.nets.policy, policy)
    for nets in (learner.nets.critics, learner.nets.targets):
        _load(nets, critics[0] + critics[1])
    learner.enable_input_slots(2)
    for k in (1, 0):
        learner.batch.load_batch(batches[k])
        learner.batch.flush()
        if k:
            learner.slot_block(k).copy_from(learner.batch.block)
    learner.update()
    out = {"policy": [_see(p) for p in learner.nets.policy.parameters()],
           "critics": [_see(p) for p in learner.nets.critics.parameters()],
           "targets": [_see(p) for p in learner.nets.targets.parameters()], "log_alpha": _see(learner.log_alpha),
           "actor_m": [_see(m) for m in learner.actor_opt.m], "critic_m": [_see(m) for m in learner.critic_opt.m]}
    return {"learner": learner, "run": _alternate(learner.replay_slot, out)}


def _prepare_ppo(case, seed):
    from ttrl_amd.algos.ppo import PPOConfig, PPOLearner, RecurrentConfig, RecurrentPPOLearner
    from ttrl_amd.spaces import ActionSpec, ObsSpec

    trunk, gru, heads, rollout = _rollout_data(case, seed)
    recurrent = RecurrentConfig(hidden_size=case["hidden"], seq_len=case["seq"]) if gru else None
    cfg = PPOConfig(lr=PPO_LR, adam_eps=EPS, minibatch_size=case["minibatch"], epochs=case["epochs"],
                    n_steps=case["steps"], recurrent=recurrent)
    learner = (RecurrentPPOLearner if gru else PPOLearner)(
        ObsSpec.image((case["channels"], case["frame"], case["frame"])), ActionSpec.discrete(case["actions"]),
        _device(), cfg=cfg, seed=seed)
    _load(learner.net, trunk + gru + heads)
    steps = learner.load_rollout(rollout)
    learner.begin_update()
    out = _adam_state(learner.optimizer)

    def run():
        learner.run_update(steps)
        return out

    return {"learner": learner, "run": run}


def _block_step(module, inputs, forward):
    """A captured forward and backward of `module` under a loss, without an optimizer."""
    from ttrl_amd.engine.step import TrainStep

    made = {}

    def body(tensors):
        module.zero_grad()
        for t in tensors.values():
            t.zero_grad()
        made["out"], loss = forward(tensors)
        loss.backward()
        return {}

    step = TrainStep(body, inputs, _device(), mode="graph")
    step.run()
    out = {"out": _see(made["out"]), "grads": [_see(p.grad) for p in module.parameters()],
           "dx": [_see(t.grad) for t in inputs.values() if t.requires_grad]}

    def run():
        step.replay()
        return out

    return {"step": step, "made": made, "run": run}


def _tensor(array, grad=False, dtype=np.float32):
    from ttrl_amd.engine.autograd import Tensor

    return Tensor.from_numpy(array, _device(), requires_grad=grad, dtype=dtype)


def _prepare_conv(case, seed):
    from ttrl_amd.engine.conv import Conv2d
    from ttrl_amd.engine.ops import mul, sum_all

    weights, x, dy = _conv_data(case, seed)
    frames, size = case["frames"], case["size"]
    net = Conv2d((case["channels"], size, size), case["out"], case["kernel"], _device(), batch=case["batch"],
                 stride=case["stride"], input_scale=1.0 / 255.0 if frames else 1.0, needs_input_grad=not frames,
                 input_layout="nchw_u8" if frames else "nhwc")
    net.load_state_dict({"weight": weights[0], "bias": weights[1]})

    def forward(t):
        y = net(t["x"])
        return y, sum_all(mul(y, t["dy"]))

    return _block_step(net, {"x": _tensor(x, not frames, x.dtype), "dy": _tensor(dy)}, forward)


def _prepare_linear(case, seed):
    from ttrl_amd.engine.layers import Linear
    from ttrl_amd.engine.ops import mean_all, square, sub

    weights, x, target = _linear_data(case, seed)
    net = Linear(case["in"], case["out"], _device())
    _load(net, weights)

    def forward(t):
        y = net(t["x"])
        return y, mean_all(square(sub(y, t["target"])))

    return _block_step(net, {"x": _tensor(x, True), "target": _tensor(target)}, forward)


def _prepare_gru(case, seed):
    from ttrl_amd.engine.ops import mul, sum_all
    from ttrl_amd.engine.recurrent import GRU

    weights, x, h0, done, dy = _gru_data(case, seed)
    net = GRU(case["in"], case["hidden"], _device())
    _load(net, weights)

    def forward(t):
        y, _ = net(t["x"], t["h0"], t["done"])
        return y, sum_all(mul(y, t["dy"]))

    return _block_step(net, {"x": _tensor(x, True), "h0": _tensor(h0, True), "done": _tensor(done), "dy": _tensor(dy)},
                       forward)


def _prepare_replay(case, seed):
    from ttrl_amd.buffers import PriorityConfig, ReplayBuffer
    from ttrl_amd.engine.tensor import DeviceArray
    from ttrl_amd.spaces import ActionSpec, ObsSpec

    base, f, steps = _replay_data(case, seed)
    lanes, n, dev = case["lanes"], case["batch"], _device()
    spec = ObsSpec.image(base.shape[2:])
    buf = ReplayBuffer(spec, ActionSpec.discrete(6), dev, capacity=case["capacity"], n_envs=lanes,
                       n_step=case["n_step"], gamma=0.99, seed=seed, priority=PriorityConfig())
    for s in range(0, steps, 64):
        e = min(s + 64, steps)
        frames = base[:e - s] ^ np.uint8(s // 64 & 255)  # every block of steps its own frames
        ends = f["ends"][s:e]
        buf.add_steps(frames, f["actions"][s:e], f["rewards"][s:e], ends, final_obs=frames)
    for lane in range(lanes):
        for c in range(0, steps, 512):
            cols = np.arange(c, min(c + 512, steps))
            buf.update_priorities(np.full(cols.size, lane), cols, f["priorities"][lane, cols])
    # the buffers a learner binds; a draw fills them in place
    sink = {k: DeviceArray(dev, (n,) + base.shape[2:], np.uint8) for k in ("obs", "next_obs")}
    sink["actions_onehot"] = DeviceArray(dev, (n, 6))
    sink.update({k: DeviceArray(dev, (n, 1)) for k in ("rewards", "dones", "discounts", "weights")})
    out = {k: _see(v) for k, v in sink.items()}

    def run():
        buf.sample(n, beta=0.5, out=sink)
        return out

    return {"buffer": buf, "sink": sink, "run": run}


def prepare(case: dict, seed: int):
    kind = "ppo" if case["kind"] == "rppo" else case["kind"]
    return globals()["_prepare_" + kind](case, seed)


def run(state):
    return state["run"]()


# ---------------------------------------------------------- float64 twins ---

def _conv(x, w, b, stride):
    o, _, k, _ = w.shape
    side = (x.shape[-1] - k) // stride + 1
    y = torch.matmul(w.reshape(o, -1), F.unfold(x, k, stride=stride)) + b.reshape(1, o, 1)
    return y.reshape(x.shape[0], o, side, side)


def _encode(p, frames):
    """The image encoder: p = four (weight, bias) pairs; -> (B, 512) features."""
    x = frames.to(p[0].dtype) * FRAME_SCALE
    for i, (_, _, stride) in enumerate(TOWER):
        x = torch.relu(_conv(x, p[2 * i], p[2 * i + 1], stride))
    return torch.relu(x.permute(0, 2, 3, 1).reshape(x.shape[0], -1) @ p[6] + p[7])


def _dense(p, x, relu_last=False):
    for i in range(0, len(p), 2):
        x = x @ p[i] + p[i + 1]
        if relu_last or i + 2 < len(p):
            x = torch.relu(x)
    return x


def _unroll(p, x, h, done):
    w_ih, w_hh, b_ih, b_hh = p
    H, gi, out = w_hh.shape[0], x @ w_ih + b_ih, []
    for t in range(x.shape[0]):
        h = h * (1.0 - done[t])
        gh = h @ w_hh + b_hh
        r, z = torch.sigmoid(gi[t, :, :2 * H] + gh[:, :2 * H]).split(H, -1)
        n = torch.tanh(gi[t, :, 2 * H:] + r * gh[:, 2 * H:])
        h = (1.0 - z) * n + z * h
        out.append(h)
    return torch.stack(out)


def _f64(arrays, grad=True) -> list:
    return [torch.from_numpy(a).cuda().double().requires_grad_(grad) for a in arrays]


def _d(a):
    return torch.from_numpy(np.asarray(a)).cuda().double()


def _layout(tensors) -> list:
    """Convolution weights in the package's storage order, [patch][out]; the rest as they are."""
    out = []
    for t in tensors:
        if t.dim() == 4 and t.shape[-1] == TOWER[0][1]:  # the first layer: patch order (c, kh, kw)
            t = t.reshape(t.shape[0], -1).T
        elif t.dim() == 4 and t.shape[0] > 1:
            t = t.permute(2, 3, 1, 0).reshape(-1, t.shape[0])
        out.append(t.detach())
    return out


class _Adam:
    """Adam with m and v stored over (1 - beta), as the package stores them."""

    def __init__(self, params, lr, eps):
        self.p, self.lr, self.eps, self.t = params, lr, eps, 0
        self.m = [torch.zeros_like(p) for p in params]
        self.v = [torch.zeros_like(p) for p in params]

    def step(self, grads):
        self.t += 1
        with torch.no_grad():
            for p, g, m, v in zip(self.p, grads, self.m, self.v):
                m.mul_(B1).add_(g)
                v.mul_(B2).add_(g * g)
                mh = m * (1 - B1) / (1 - B1 ** self.t)
                vh = v * (1 - B2) / (1 - B2 ** self.t)
                p -= self.lr * mh / (vh.sqrt() + self.eps)

    def state(self) -> dict:
        # The moments of a whole network follow its gates and clips, which
        # rounding may decide either way (above); the layers' own cases hold
        # the gradients' arithmetic.
        none = [None] * len(self.p)
        return {"params": _layout(self.p), "m": none, "v": none}


def _exact_act_greedy(case, seed):
    rng = np.random.default_rng(seed)
    n, shape = case["lanes"], (case["channels"], case["frame"], case["frame"])
    p = _f64(_weights(rng, _tower_shapes(*shape[:2]) + [(512, case["actions"])]), False)
    obs = torch.from_numpy(rng.integers(0, 256, (n,) + shape, dtype=np.uint8)).cuda()
    return {"actions": None, "q": _encode(p[:8], obs) @ p[8] + p[9]}


def _sample(p, obs, noise):
    h = _dense(p[:4], obs, relu_last=True)
    mean, log_std = h @ p[4] + p[5], (h @ p[6] + p[7]).clamp(-20.0, 2.0)
    u = mean + log_std.exp() * noise
    logp = (-0.5 * noise * noise - log_std - 0.5 * math.log(2 * math.pi)
            - 2.0 * (math.log(2.0) - u - F.softplus(-2.0 * u))).sum(-1)
    return torch.tanh(u), logp


def _exact_act_squashed(case, seed):
    rng = np.random.default_rng(seed)
    n, O, A, H = case["lanes"], case["obs"], case["act"], case["hidden"]
    p = _f64(_weights(rng, _mlp_shapes(O, H, H) + [(H, A), (H, A)]), False)
    obs, noise = (_d(rng.standard_normal((n, k)).astype(np.float32)) for k in (O, A))
    action, logp = _sample(p, obs, noise)
    return {"action": action, "logp": logp}


def _exact_dqn(case, seed):
    online, target, batches = _dqn_data(case, seed)
    p, tp = _f64(online), _f64(target, False)
    opt = _Adam(p, DQN_LR, DQN_EPS)
    for b in batches:
        obs, nxt = (torch.from_numpy(b[k]).cuda() for k in ("obs", "next_obs"))
        rows = torch.arange(case["batch"], device="cuda")
        q = (_encode(p[:8], obs) @ p[8] + p[9])[rows, torch.from_numpy(b["actions"]).cuda()]
        with torch.no_grad():
            tq = _encode(tp[:8], nxt) @ tp[8] + tp[9]
            pick = _encode(p[:8], nxt) @ p[8] + p[9] if case["double"] else tq
            y = _d(b["rewards"]) + _d(b["discounts"]) * (1 - _d(b["dones"])) * tq[rows, pick.argmax(-1)]
        loss = (_d(b["is_weights"]) * F.huber_loss(q, y, reduction="none")).mean()
        grads = torch.autograd.grad(loss, p)
        opt.step(grads)
    out = opt.state()
    if case["read"]:
        out["metrics"] = {"loss": loss.detach(), "mean_q": q.detach().mean(), "td_abs": (q - y).detach().abs(),
                          "grad_sq": None}
    return out


def _exact_sac(case, seed):
    policy, critics, batches = _sac_data(case, seed)
    pol, cr, tg = _f64(policy), _f64(critics[0] + critics[1]), _f64(critics[0] + critics[1], False)
    log_alpha = torch.zeros(1, device="cuda", dtype=torch.float64, requires_grad=True)
    actor, critic, temp = _Adam(pol, SAC_LR, EPS), _Adam(cr, SAC_LR, EPS), _Adam([log_alpha], SAC_LR, EPS)

    def both(p, obs, action):
        x = torch.cat([obs, action], -1)
        return _dense(p[:6], x).reshape(-1), _dense(p[6:], x).reshape(-1)

    for b in batches:
        t = {k: _d(v) for k, v in b.items()}
        with torch.no_grad():
            a2, lp2 = _sample(pol, t["next_obs"], t["next_noise"])
            soft = torch.minimum(*both(tg, t["next_obs"], a2)) - log_alpha.exp() * lp2
            y = t["rewards"] + t["discounts"] * (1 - t["dones"]) * soft
        loss = sum(0.5 * ((q - y) ** 2).mean() for q in both(cr, t["obs"], t["actions"]))
        critic.step(torch.autograd.grad(loss, cr))
        a, lp = _sample(pol, t["obs"], t["noise"])
        loss = (log_alpha.detach().exp() * lp - torch.minimum(*both(cr, t["obs"], a))).mean()
        grads = torch.autograd.grad(loss, pol)
        d_alpha = -(lp.detach() - case["act"]).mean().reshape(1)
        actor.step(grads)
        temp.step([d_alpha])
        with torch.no_grad():
            for x, c in zip(tg, cr):
                x.mul_(1 - 0.005).add_(0.005 * c)
    return {"policy": [x.detach() for x in pol], "critics": [x.detach() for x in cr], "targets": tg,
            "log_alpha": log_alpha.detach(), "actor_m": [None] * len(pol), "critic_m": [None] * len(cr)}


def _exact_ppo(case, seed):
    trunk, gru, heads, r = _rollout_data(case, seed)
    T, N, mb, A = case["steps"], case["envs"], case["minibatch"], case["actions"]
    p = _f64(trunk + gru + heads)
    adv, last, nv = np.zeros((T, N)), np.zeros(N), r["last_values"].astype(np.float64)
    for t in range(T - 1, -1, -1):
        alive = 1.0 - r["dones"][t]
        last = r["rewards"][t] + 0.99 * nv * alive - r["values"][t] + 0.99 * 0.95 * alive * last
        adv[t], nv = last, r["values"][t].astype(np.float64)
    flat = {"adv": _d((adv - adv.mean()) / (adv.std() + 1e-8)).reshape(-1), "ret": _d(adv + r["values"]).reshape(-1),
            "value": _d(r["values"]).reshape(-1), "logp": _d(r["logp"]).reshape(-1),
            "action": torch.from_numpy(r["actions"].reshape(-1)).cuda()}
    obs = torch.from_numpy(r["obs"].reshape((T * N,) + r["obs"].shape[2:])).cuda()
    rng, opt = np.random.default_rng(seed), _Adam(p, PPO_LR, EPS)
    L = case.get("seq", 1)
    S, units = mb // L, T // L * N
    for _ in range(case["epochs"]):
        perm = rng.permutation(units)
        for k in range(0, units // S * S, S):
            ids = perm[k:k + S]
            ch, lane = ids // N, ids % N
            rows = (((ch[None] * L + np.arange(L)[:, None]) * N + lane[None]).reshape(-1))
            at = torch.from_numpy(rows).cuda()
            h = _encode(p[:8], obs[at])
            if gru:
                starts = _d(r["starts"].reshape(-1)[rows]).reshape(L, S, 1)
                h0 = _d(r["hidden"].reshape(-1, case["hidden"])[ids])
                h = _unroll(p[8:12], h.reshape(L, S, -1), h0, starts).reshape(L * S, -1)
            logp = torch.log_softmax(h @ p[-4] + p[-3], -1)
            v = (h @ p[-2] + p[-1]).reshape(-1)
            b = {n: x[at] for n, x in flat.items()}
            ratio = (logp.gather(1, b["action"][:, None]).reshape(-1) - b["logp"]).exp()
            gain = torch.minimum(ratio * b["adv"], ratio.clamp(0.9, 1.1) * b["adv"]).mean()
            near = b["value"] + (v - b["value"]).clamp(-0.1, 0.1)
            value = 0.5 * torch.maximum((v - b["ret"]) ** 2, (near - b["ret"]) ** 2).mean()
            entropy = -(logp.exp() * logp).sum(-1).mean()
            grads = torch.autograd.grad(-gain + 0.5 * value - 0.01 * entropy, p)
            norm = math.sqrt(sum(float((g * g).sum()) for g in grads))
            scale = 0.5 / (norm + 1e-6) if norm > 0.5 else 1.0
            opt.step([g * scale for g in grads])
    return opt.state()


def _exact_conv(case, seed):
    weights, x, dy = _conv_data(case, seed)
    p, x = _f64(weights), torch.from_numpy(x).cuda().double()
    x = x * FRAME_SCALE if case["frames"] else x.requires_grad_()
    y = _conv(x if case["frames"] else x.permute(0, 3, 1, 2), p[0], p[1], case["stride"])
    y = y.permute(0, 2, 3, 1).reshape(1, 1, -1, case["out"])
    grads = torch.autograd.grad((y * _d(dy)).sum(), p if case["frames"] else p + [x])
    w = grads[0]
    w = w.reshape(w.shape[0], -1).T if case["frames"] else w.permute(2, 3, 1, 0).reshape(-1, w.shape[0])
    return {"out": y.detach(), "grads": [w, grads[1]], "dx": list(grads[2:])}


def _exact_linear(case, seed):
    weights, x, target = _linear_data(case, seed)
    p, x = _f64(weights), _d(x).requires_grad_()
    y = x @ p[0] + p[1]
    *grads, dx = torch.autograd.grad(((y - _d(target)) ** 2).mean(), p + [x])
    return {"out": y.detach(), "grads": grads, "dx": [dx]}


def _exact_gru(case, seed):
    weights, x, h0, done, dy = _gru_data(case, seed)
    p, x, h0 = _f64(weights), _d(x).requires_grad_(), _d(h0).requires_grad_()
    y = _unroll(p, x, h0, _d(done))
    *grads, dx, dh = torch.autograd.grad((y * _d(dy)).sum(), p + [x, h0])
    return {"out": y.detach(), "grads": grads, "dx": [dx, dh]}


def _exact_replay(case, seed):
    """The first draw's numbers: n-step returns, discounts and importance weights."""
    _, f, steps = _replay_data(case, seed)
    rng, n, k = np.random.default_rng(seed), case["batch"], case["n_step"]
    count = steps - k
    w = (f["priorities"] + 1e-6) ** 0.6
    sums = w[:, :count].sum(1)
    quota = rng.multinomial(n, sums / sums.sum())
    lanes = np.repeat(np.arange(case["lanes"]), quota)
    u, cols = rng.random(n), np.zeros(n, np.int64)
    cdf = np.cumsum(w[:, :count], 1)
    for i, lane in enumerate(lanes):
        cols[i] = min(int(np.searchsorted(cdf[lane], u[i] * cdf[lane, -1], side="right")), count - 1)
    rewards, discounts, dones = np.zeros((n, 1)), np.ones((n, 1)), np.zeros((n, 1))
    for i, (lane, col) in enumerate(zip(lanes, cols)):
        for j in range(col, col + k):
            rewards[i] += discounts[i] * f["rewards"][j, lane].astype(np.float64)
            discounts[i] *= 0.99
            if f["ends"][j, lane]:
                dones[i] = 1.0
                break
    weights = (case["lanes"] * count * w[lanes, cols] / sums.sum()) ** -0.5
    return {"obs": None, "next_obs": None, "actions_onehot": None, "rewards": rewards, "dones": dones,
            "discounts": discounts, "weights": (weights / weights.max()).reshape(n, 1)}


def exact(case: dict, seed: int):
    kind = "ppo" if case["kind"] == "rppo" else case["kind"]
    return globals()["_exact_" + kind](case, seed)


# ------------------------------------------------------ work, tolerances ----

def _macs(case) -> tuple:
    """Multiply-accumulates a sample of the image encoder takes: all of it, its first layer."""
    macs, c = [], case["channels"]
    for (o, k, _), side in zip(TOWER, _sizes(case["frame"])):
        macs.append(side * side * o * c * k * k)
        c = o
    macs.append(_sizes(case["frame"])[-1] ** 2 * c * 512)
    return sum(macs), macs[0]


def _count(shapes) -> int:
    return sum(int(np.prod(s)) + (s[0] if len(s) == 4 else s[1]) for s in shapes)


def work(case: dict) -> dict:
    kind = case["kind"]
    if "frame" in case and kind != "replay":
        frame = case["channels"] * case["frame"] ** 2
        total, first = _macs(case)
        n = _count(_tower_shapes(case["channels"], case["frame"]))
    if kind == "act_greedy":
        macs = total + 512 * case["actions"]
        return {"bytes": case["lanes"] * frame + 4 * (n + 512 * case["actions"]), "flops": 2 * case["lanes"] * macs}
    if kind == "act_squashed":
        n = _count(_mlp_shapes(case["obs"], case["hidden"], case["hidden"], 2 * case["act"]))
        return {"bytes": 4 * (n + case["lanes"] * (case["obs"] + 2 * case["act"])), "flops": 2 * case["lanes"] * n}
    if kind == "dqn":
        # three (or two) forwards, weight gradients, input gradients but the first layer's, Adam
        total, n = total + 512 * case["actions"], n + 512 * case["actions"]
        sweeps = (5 if case["double"] else 4) * total - first
        return {"bytes": 2 * case["batch"] * frame + 28 * n, "flops": 2 * case["batch"] * sweeps}
    if kind == "sac":
        O, A, H = case["obs"], case["act"], case["hidden"]
        pol, crit = _count(_mlp_shapes(O, H, H, 2 * A)), _count(_mlp_shapes(O + A, H, H, 1))
        # forwards: policy on s and s', target, online and stepped critics; backwards of critics and policy
        macs = 2 * pol + 6 * crit + 4 * crit + 2 * crit + 2 * pol
        floats = 24 * pol + 2 * 32 * crit + 4 * case["batch"] * (2 * O + 3 * A + 3)
        return {"bytes": floats, "flops": 2 * case["batch"] * macs}
    if kind in ("ppo", "rppo"):
        H = case.get("hidden", 512)
        per = 3 * total - first + 3 * H * (case["actions"] + 1)
        n += H * (case["actions"] + 1)
        if kind == "rppo":
            per += 3 * 3 * H * (512 + H)
            n += 3 * H * (512 + H)
        L = case.get("seq", 1)
        steps = case["epochs"] * (case["steps"] // L * case["envs"] // (case["minibatch"] // L))
        return {"bytes": steps * (case["minibatch"] * frame + 24 * n), "flops": 2 * steps * case["minibatch"] * per}
    if kind == "conv":
        side = (case["size"] - case["kernel"]) // case["stride"] + 1
        n = _count([(case["out"], case["channels"], case["kernel"], case["kernel"])])
        x, y = case["channels"] * case["size"] ** 2, case["out"] * side * side
        read = x if case["frames"] else 8 * x
        return {"bytes": case["batch"] * (read + 8 * y) + 8 * n,
                "flops": 2 * case["batch"] * side * side * n * (2 if case["frames"] else 3)}
    if kind == "linear":
        n = _count([(case["in"], case["out"])])
        return {"bytes": 8 * n + 8 * case["rows"] * (case["in"] + case["out"]), "flops": 6 * case["rows"] * n}
    if kind == "gru":
        n, rows = 3 * case["hidden"] * (case["in"] + case["hidden"] + 2), case["steps"] * case["batch"]
        return {"bytes": 8 * n + 8 * rows * (case["in"] + case["hidden"]), "flops": 6 * rows * n}
    frame = 4 * case["frame"] ** 2
    return {"bytes": 4 * case["batch"] * frame + 8 * case["capacity"], "flops": case["capacity"]}


def tolerance(case: dict):
    """About four times what two float32 orders of the same sums show
    against float64 over the drawn ranges."""
    if case["kind"] in ("dqn", "sac", "ppo", "rppo"):  # 1.4e-3 and 5e-3 where a gate flips, else 1e-6
        return {"rel": 5e-3, "max": 2e-2}
    if case["kind"] == "replay":
        return {"rel": 2e-7, "max": 5e-7}
    return {"rel": 4e-6, "max": 2e-5, "differ": 0.01 if case["kind"] == "act_greedy" else 0.0}
