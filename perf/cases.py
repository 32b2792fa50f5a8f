"""Timed cases: what a program built on qqtsim has the GPU do.

`listed()` holds the cases, `draw(rng)` gives more of the same ranges,
`prepare(case, seed)` builds what the program holds before the call (on the
GPU, from the seed alone), `run(state)` makes one pass through the public
entry points, `work(case)` states the bytes and operations of one pass,
`tolerance(case)` what another correct implementation may differ by, and
`exact(case, seed)` the same outputs from plain float64 torch.

The kinds, by use:

  step      `HipBatchedSim.step` + `observe` + `legal_mask`: a caller that
            drives the sim itself (evaluation, small batches, other grids)
  tick      `TickLoop.launch_tick`: the sim alone at rollout sizes, injected
            actions, auto-reset (the bomb-stress workload)
  rollout   one `Rollout.step` of self-play with the mlp policy (collection)
  versus    one `Rollout.step` of the mlp learner against the astar bot
  lroll     one `LstmRollout.step`: lstm learner against the astar bot
  act       `act_pair` of the mlp or cnn policy on a batch of observations
  lforward  `HipLstmActorCritic.forward`: one frame of a batch of sequences
  forward   `HipActorCritic.forward` over a slab of observations (evaluation)
  grads     `HipMlpActorCritic.ppo_grads` of one minibatch of rows of a
            rollout buffer (forward, loss and backward of a PPO update)
  lupdate   `ppo_update` of the lstm learner over a rollout buffer of
            sequences (one epoch, one minibatch: truncated BPTT, Adam)
"""

import math
import os
import sys

import torch
import torch.utils.checkpoint

# the package lives in a folder whose name is not an identifier
_PKG = os.path.join(os.getcwd(), "qqt-gpu-sim_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from qqtsim import (BOMB_STRESS_40, CORRIDOR_70, HipActorCritic, HipAstarBot, HipBatchedSim,  # noqa: E402
                    HipCnnActorCritic, HipLstmActorCritic, HipMlpActorCritic, HipRolloutBuffer,
                    LstmLearner, LstmRollout, MapSpec, PPOConfig, Rollout, corridor_training_config,
                    ppo_update, reference_init)
from qqtsim.rollout import TickLoop  # noqa: E402

MAPS = {"bricks": CORRIDOR_70, "stress": BOMB_STRESS_40, "open": MapSpec(kind="open"),
        "reference": MapSpec(kind="reference")}
GRIDS = ((13, 2), (13, 2), (13, 2), (13, 3), (13, 4), (9, 2), (7, 2))   # (height = width, players)
WARM = 36            # ticks before a measured state: bombs of the first ticks have exploded


# ------------------------------------------------------------------ cases
def listed():
    return [
        # the smallest calls: a debugging or evaluation loop over few envs
        dict(name="step_64", kind="step", n=64, grid=13, players=2, maps="bricks"),
        # both players of a handful of envs (serving, an odd batch)
        dict(name="act_mlp_37", kind="act", net="mlp", n=37),
        # one frame of a ragged batch of lstm sequences
        dict(name="lforward_1021", kind="lforward", n=1021),
        # four players on a ragged batch: the sim at a fifth of a rollout
        dict(name="tick_1021_p4", kind="tick", n=1021, grid=13, players=4, maps="stress"),
        # the bomb-stress workload
        dict(name="tick_16384", kind="tick", n=16384, grid=13, players=2, maps="stress"),
        # self-play collection at the training batch
        dict(name="rollout_5632", kind="rollout", n=5632, maps="bricks"),
        # the learner against the rule bot, approach / flee modes on
        dict(name="versus_5632", kind="versus", n=5632, maps="bricks", modes=True),
        # the lstm learner against the rule bot
        dict(name="lroll_5632", kind="lroll", n=5632, maps="bricks"),
        # the cnn policy for both players at the training batch
        dict(name="act_cnn_5632", kind="act", net="cnn", n=5632),
        # evaluation forward over 128 ticks of 32768 envs
        dict(name="forward_4M", kind="forward", n=32768, steps=128),
        # one minibatch of four of a 5632 x 128 PPO update
        dict(name="grads_180224", kind="grads", n=5632, steps=128, rows=180224),
        # the lstm update over a small buffer (at the training batch the
        # convolution library's search for one new shape takes minutes)
        dict(name="lupdate_256x32", kind="lupdate", n=256, steps=32),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("step", "tick", "rollout", "versus", "lroll", "act", "act", "lforward",
                       "forward", "grads", "lupdate"))
    if kind in ("step", "tick"):
        grid, players = rng.choice(GRIDS)
        return dict(kind=kind, n=_log_int(rng, 1, 16384), grid=grid, players=players,
                    maps=rng.choice(sorted(MAPS)) if grid == 13 and players == 2
                    else rng.choice(("bricks", "open", "stress")))
    if kind == "rollout":
        return dict(kind=kind, n=_log_int(rng, 16, 16384),
                    maps=rng.choice(("bricks", "reference")))
    if kind == "versus":
        return dict(kind=kind, n=_log_int(rng, 16, 16384), maps=rng.choice(("bricks", "reference")),
                    modes=rng.random() < 0.5)
    if kind == "lroll":
        return dict(kind=kind, n=_log_int(rng, 16, 8192), maps=rng.choice(("bricks", "reference")))
    if kind == "act":
        net = rng.choice(("mlp", "cnn"))
        return dict(kind=kind, net=net, n=_log_int(rng, 1, 16384 if net == "mlp" else 8192))
    if kind == "lforward":
        return dict(kind=kind, n=_log_int(rng, 1, 16384))
    if kind == "forward":
        return dict(kind=kind, n=_log_int(rng, 64, 32768), steps=_log_int(rng, 8, 128))
    if kind == "grads":
        n, steps = _log_int(rng, 64, 5632), _log_int(rng, 16, 128)
        return dict(kind=kind, n=n, steps=steps, rows=max(1, n * steps // rng.choice((1, 2, 4, 8))))
    return dict(kind=kind, n=_log_int(rng, 16, 256), steps=_log_int(rng, 8, 32))


# ----------------------------------------------------------------- inputs
def _dev():
    return torch.device("cuda:0")


def _gen(seed):
    return torch.Generator(device=_dev()).manual_seed(int(seed) * 7919 + 13)


def _cfg(case):
    g, p = case.get("grid", 13), case.get("players", 2)
    if (g, p) == (13, 2):
        return corridor_training_config()
    return corridor_training_config(height=g, width=g, n_players=p,
                                    corridor_width=min(g - 2, max(5, 2 * p - 1)),
                                    top_wall_rows=min(4, g - 3))


def _random_actions(steps, n, p, gen):
    """Uniform moves, a bomb with probability 1/2: what a policy at its
    initial weights plays."""
    a = torch.randint(0, 5, (steps, n, p, 2), generator=gen, device=_dev(), dtype=torch.int8)
    a[..., 1] = torch.randint(0, 2, (steps, n, p), generator=gen, device=_dev(), dtype=torch.int8)
    return a


def _warm_sim(case, seed, gen):
    """A sim in mid-game: `WARM` ticks of random actions."""
    cfg = _cfg(case)
    sim = HipBatchedSim(cfg, case["n"], device=_dev(), seed=seed, map_spec=MAPS[case["maps"]])
    loop = TickLoop(sim)
    for a in _random_actions(WARM, case["n"], cfg.n_players, gen):
        loop.launch_tick(a)
    return sim, loop


def _slab(n, steps, seed, gen):
    """(steps, n, C, H, W) observations of random play, as a rollout stores them."""
    sim, loop = _warm_sim(dict(n=n, maps="bricks"), seed, gen)
    out = torch.empty((steps, n) + tuple(sim.cfg.obs_shape), dtype=torch.float16, device=_dev())
    for t in range(steps):
        out[t].copy_(sim.observe())
        loop.launch_tick(_random_actions(1, n, 2, gen)[0])
    return out


def _weights(arch, seed):
    """The reference's initial weights with the policy heads' outputs at a
    trained scale, so that logits and their gradients are not all near zero."""
    sd = reference_init(seed=seed, arch=arch)
    g = torch.Generator().manual_seed(int(seed) + 5)
    for k in ("move_head.2.weight", "bomb_head.2.weight"):
        sd[k] = sd[k] + 0.1 * torch.randn(sd[k].shape, generator=g)
    for k in sd:
        if k.endswith("bias"):
            sd[k] = sd[k] + 0.02 * torch.randn(sd[k].shape, generator=g)
    return sd


def _legal_actions(mm, bm, gen):
    """Uniform legal (moves, bombs) and their log-probability."""
    r = torch.rand(mm.shape, generator=gen, device=_dev()).masked_fill(~mm, -1.0)
    s = torch.rand(bm.shape, generator=gen, device=_dev()).masked_fill(~bm, -1.0)
    act = torch.stack([r.argmax(-1), s.argmax(-1)], -1)
    return act, -(mm.sum(-1).float().log() + bm.sum(-1).float().log())


def prepare(case, seed):
    kind, n, dev = case["kind"], case["n"], _dev()
    gen = _gen(seed)
    if kind in ("step", "tick"):
        sim, loop = _warm_sim(case, seed, gen)
        acts = list(_random_actions(16, n, sim.cfg.n_players, gen))
        if kind == "step":
            acts = [a.long() for a in acts]
        return dict(case=case, sim=sim, loop=loop, actions=acts, at=0)
    if kind in ("rollout", "versus"):
        sim, _ = _warm_sim(case, seed, gen)
        net = HipActorCritic(_weights("mlp", seed), device=dev, seed=seed)
        bot = HipAstarBot(sim, 1, mode=case["modes"]) if kind == "versus" else None
        return dict(case=case, sim=sim, roll=Rollout(sim, net, bot))
    if kind == "lroll":
        sim, _ = _warm_sim(case, seed, gen)
        net = HipLstmActorCritic(_weights("lstm", seed), device=dev, seed=seed)
        roll = LstmRollout(sim, net, HipAstarBot(sim, 1))
        roll.h.normal_(0.0, 0.3, generator=gen)
        roll.c.normal_(0.0, 0.6, generator=gen)
        return dict(case=case, sim=sim, roll=roll)
    if kind == "act":
        sim, _ = _warm_sim(dict(n=n, maps="bricks"), seed, gen)
        cls = HipActorCritic if case["net"] == "mlp" else HipCnnActorCritic
        sd = _weights(case["net"], seed)
        mm, bm = sim.legal_mask()
        return dict(case=case, net=cls(sd, device=dev, seed=seed), weights=sd, obs=sim.observe(),
                    mm=mm, bm=bm)
    if kind == "lforward":
        sim, _ = _warm_sim(dict(n=n, maps="bricks"), seed, gen)
        sd = _weights("lstm", seed)
        h = 0.3 * torch.randn((1, n, 128), generator=gen, device=dev)
        c = 0.6 * torch.randn((1, n, 128), generator=gen, device=dev)
        return dict(case=case, net=HipLstmActorCritic(sd, device=dev, seed=seed), weights=sd,
                    feat=[f[:, 0] for f in sim.local_view_features(only_p0=True)], hidden=(h, c))
    if kind == "forward":
        sd = _weights("mlp", seed)
        obs = _slab(n, case["steps"], seed, gen)
        return dict(case=case, net=HipActorCritic(sd, device=dev, seed=seed), weights=sd,
                    obs=obs.view(-1, *obs.shape[2:]))
    if kind == "grads":
        sd = _weights("mlp", seed)
        sim, loop = _warm_sim(dict(n=n, maps="bricks"), seed, gen)
        t, total = case["steps"], case["steps"] * n
        s = dict(case=case, weights=sd, net=HipMlpActorCritic(device=dev, state_dict=sd),
                 cfg=PPOConfig(),
                 obs=torch.empty((t, n) + tuple(sim.cfg.obs_shape), dtype=torch.float16, device=dev),
                 mm=torch.empty((t, n, 5), dtype=torch.uint8, device=dev),
                 bm=torch.empty((t, n, 2), dtype=torch.uint8, device=dev))
        for i in range(t):
            s["obs"][i].copy_(sim.observe())
            mm, bm = sim.legal_mask()
            s["mm"][i].copy_(mm[:, 0])
            s["bm"][i].copy_(bm[:, 0])
            loop.launch_tick(_random_actions(1, n, 2, gen)[0])
        for k in ("obs", "mm", "bm"):
            s[k] = s[k].view(total, *s[k].shape[2:])
        act, lp = _legal_actions(s["mm"].bool(), s["bm"].bool(), gen)
        f = lambda scale: scale * torch.randn((total,), generator=gen, device=dev)  # noqa: E731
        s.update(act=act, old_logp=lp + f(0.1), adv=f(1.0), ret=f(1.0), old_val=f(0.5),
                 rows=torch.randperm(total, generator=gen, device=dev)[:case["rows"]].contiguous())
        return s
    # lupdate
    sd = _weights("lstm", seed)
    learner = LstmLearner(state_dict=sd).to(dev)
    sim, loop = _warm_sim(dict(n=n, maps="bricks"), seed, gen)
    buf = HipRolloutBuffer(case["steps"], n, sim.cfg.obs_shape, dev, arch="lstm")
    for _ in range(case["steps"]):
        mm, bm = sim.legal_mask()
        act, lp = _legal_actions(mm[:, 0], bm[:, 0], gen)
        feat = [x[:, 0] for x in sim.local_view_features(only_p0=True)]
        a = _random_actions(1, n, 2, gen)[0]
        a[:, 0] = act.to(torch.int8)
        mm, bm = mm[:, 0].clone(), bm[:, 0].clone()
        loop.launch_tick(a)
        noise = torch.randn((4, n), generator=gen, device=dev)
        buf.add(feat, mm, bm, act, lp + 0.1 * noise[0], 0.5 * noise[1], 0.3 * noise[2],
                torch.rand((n,), generator=gen, device=dev) < 0.01, noise[3] > 2.0)
    opt = torch.optim.Adam(learner.parameters(), lr=PPOConfig.lr)
    return dict(case=case, weights=sd, learner=learner, opt=opt, buf=buf,
                last_val=0.5 * torch.randn((n,), generator=gen, device=dev),
                cfg=PPOConfig(rollout_steps=case["steps"], epochs=1, minibatches=1))


# ------------------------------------------------------------------- pass
def _bits(x):
    """Float16 / float32 values as whole numbers of their bits: a sim's
    outputs are equal or they belong to an env whose sampled action fell on
    the other side of a tie."""
    return x.view(torch.int16 if x.dtype == torch.float16 else torch.int32)


def run(s):
    kind = s["case"]["kind"]
    if kind in ("step", "tick"):
        sim, a = s["sim"], s["actions"][s["at"] % 16]
        s["at"] += 1
        if kind == "tick":
            s["loop"].launch_tick(a)
            mm, bm = sim.legal_mask()
            return dict(obs=sim.observe(), mm=mm, bm=bm)
        reward, done, info = sim.step(a)
        mm, bm = sim.legal_mask()
        return dict(obs=sim.observe(), mm=mm, bm=bm, reward=reward, done=done, died=info["died"],
                    n_alive=info["n_alive"], winner=info["winner"])
    if kind in ("rollout", "versus", "lroll"):
        r = s["roll"]
        r.step()
        out = dict(actions=r.actions, logp=r.logp, value=r.value, obs=_bits(s["sim"].observe()),
                   reward=_bits(r.reward), done=r.done)
        if kind == "versus":     # player 1's columns are the bot's: the policy leaves them
            out.update(logp=r.logp[:, 0], value=r.value[:, 0])
        if kind == "lroll":
            out.update(logp=r.logp[:, 0], value=r.value[:, 0], h=r.h, c=r.c)
        return out
    if kind == "act":
        act, logp, value, logits = s["net"].act_pair(s["obs"], s["mm"], s["bm"], logits=True)
        return dict(actions=act, logp=logp, value=value, logits=logits)
    if kind == "lforward":
        ml, bl, v, (h, c) = s["net"].forward(s["feat"], 0, s["hidden"])
        return dict(move=ml, bomb=bl, value=v, h=h, c=c)
    if kind == "forward":
        ml, bl, v = s["net"].forward(s["obs"], 0)
        return dict(move=ml, bomb=bl, value=v)
    if kind == "grads":
        stats = s["net"].ppo_grads(s["obs"], s["mm"], s["bm"], s["act"], s["old_logp"], s["adv"],
                                   s["ret"], s["old_val"], s["cfg"], s["cfg"].entropy_coef,
                                   rows=s["rows"])
        return dict(stats=stats, grads={k: p.grad for k, p in s["net"].named_parameters()})
    stats = ppo_update(s["learner"], s["opt"], s["buf"], s["last_val"], s["cfg"],
                       s["cfg"].entropy_coef)
    return dict(stats=[stats[k] for k in sorted(stats)],
                grads={k: p.grad for k, p in s["learner"].named_parameters()},
                weights={k: p.detach() for k, p in s["learner"].named_parameters()
                         if k.startswith("lstm")})


# ------------------------------------------------------------ work and bounds
_MLP_TAIL = 128 * 128 + 128 * 192 + 5 * 64 + 2 * 64 + 64            # multiply-adds past layer 1
_CNN_MACS = 169 * (9 * (14 * 16 + 16 * 32 + 32 * 64) + 64 * 8) + 1352 * 128 + _MLP_TAIL
_LSTM_TRUNK = 49 * 9 * (14 * 32 + 32 * 64) + 576 * 128 + 60 * 64 + 64 * 32 + 5 * 16 + 16 * 8 + 168 * 256
_LSTM_MACS = _LSTM_TRUNK + 384 * 512 + 128 * 192 + 8 * 64
_LSTM_FEAT = 2 * (14 * 49 + 60 + 5)                                  # bytes of one frame's features
_K0 = 14 * 169


def _tick_bytes(case):
    g, p = case.get("grid", 13), case.get("players", 2)
    c = 5 * p + 4
    # packed cells, players and env words in and out; observation, masks, reward, done; actions in
    return case["n"] * (2 * (4 * g * g + 64 * p + 16) + 2 * c * g * g + 7 * p + 4 * p + 1 + 2 * p)


def work(case):
    kind, n = case["kind"], case["n"]
    w_mlp, w_cnn, w_lstm = 4 * 345288, 4 * 281744, 4 * 368816
    out = n * 2 * (2 + 4 + 4)                       # both players' actions, log-prob, value
    if kind in ("step", "tick"):
        return {"bytes": _tick_bytes(case), "flops": 0}
    if kind == "rollout":
        return {"bytes": _tick_bytes(case) + n * (2 * _K0 + 14) + out + w_mlp,
                "flops": 2 * 2 * n * (_K0 * 128 + _MLP_TAIL)}
    if kind == "versus":
        return {"bytes": _tick_bytes(case) + n * (2 * _K0 + 14 + 4 * 169 + 2 * 169 + 128) + out + w_mlp,
                "flops": 2 * n * (_K0 * 128 + _MLP_TAIL)}
    if kind == "lroll":
        return {"bytes": _tick_bytes(case) + n * (2 * _K0 + 14 + 4 * 169 + 128 + 4 * 512) + out + w_lstm,
                "flops": 2 * n * _LSTM_MACS}
    if kind == "act":
        return {"bytes": n * (2 * _K0 + 14 + 64 + 2 * 16 + 16) + (w_mlp if case["net"] == "mlp" else w_cnn),
                "flops": 2 * 2 * n * (_K0 * 128 + _MLP_TAIL if case["net"] == "mlp" else _CNN_MACS)}
    if kind == "lforward":
        return {"bytes": n * (_LSTM_FEAT + 4 * 512 + 32) + w_lstm, "flops": 2 * n * _LSTM_MACS}
    if kind == "forward":
        rows = n * case["steps"]
        return {"bytes": rows * (2 * _K0 + 32) + w_mlp, "flops": 2 * rows * (_K0 * 128 + _MLP_TAIL)}
    if kind == "grads":      # layer 1 forward and weight gradient, the rest also its input gradient
        return {"bytes": case["rows"] * (2 * _K0 + 8 + 7 + 16 + 16) + 2 * w_mlp,
                "flops": 2 * case["rows"] * (2 * _K0 * 128 + 3 * _MLP_TAIL)}
    rows = n * case["steps"]
    return {"bytes": rows * (_LSTM_FEAT + 16 + 7 + 24) + 6 * w_lstm,
            "flops": 2 * rows * (3 * _LSTM_MACS - 49 * 9 * 14 * 32)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("step", "tick"):
        return "exact"
    if kind in ("rollout", "versus"):
        # float16 first-layer products: logits differ by ~4e-4 between correct
        # kernels, which moves a few of 10,000 draws over a boundary
        return {"rel": 5e-3, "max": 0.9, "differ": 5e-3}
    if kind == "lroll":
        return {"rel": 1e-3, "max": 0.9, "differ": 2e-3}
    if kind == "act" and case["net"] == "mlp":
        return {"rel": 5e-3, "max": 0.9, "differ": 5e-3}
    if kind == "act":
        return {"rel": 1e-3, "max": 0.9, "differ": 2e-3}
    if kind == "lforward":
        return {"rel": 5e-6, "max": 5e-4}
    if kind == "forward":
        return {"rel": 1e-3, "max": 5e-2}
    if kind == "grads":
        return {"rel": 2e-3, "max": 0.3}
    return {"rel": 5e-4, "max": 0.1}


# ------------------------------------------------------------------ float64
# channels of the observation in the order player 0 / 1 sees them: own position
# and fuse, the opponent's, then the shared ones
_VIEW = ([0, 2, 1, 3] + list(range(4, 14)), [1, 3, 0, 2] + list(range(4, 14)))


def _f64(weights):
    return {k: v.to(_dev(), torch.float64) for k, v in weights.items()}


def _heads64(x, w):
    """Hidden features -> (n, 8): move logits, bomb logits, value."""
    outs = []
    for name in ("move_head", "bomb_head", "critic"):
        y = torch.relu(x @ w[f"{name}.0.weight"].t() + w[f"{name}.0.bias"])
        outs.append(y @ w[f"{name}.2.weight"].t() + w[f"{name}.2.bias"])
    return torch.cat(outs, -1)


def _shared64(x, w):
    ln = torch.nn.functional.layer_norm
    for i in (0, 3):
        x = x @ w[f"shared.{i}.weight"].t() + w[f"shared.{i}.bias"]
        x = torch.relu(ln(x, x.shape[-1:], w[f"shared.{i + 1}.weight"], w[f"shared.{i + 1}.bias"]))
    return x


def _mlp64(obs, w, pid):
    x = obs[:, _VIEW[pid]].double()
    return _heads64(_shared64(x.flatten(1), w), w)


def _conv64(x, w, b, pad):
    n, _, h, v = x.shape
    cols = torch.nn.functional.unfold(x, w.shape[-1], padding=pad)            # (n, c k k, h v)
    return (w.flatten(1) @ cols + b[:, None]).view(n, w.shape[0], h, v)


def _cnn64(obs, w, pid):
    x = obs[:, _VIEW[pid]].double()
    for conv, norm in (("conv0", "conv.0"), ("conv.2", "conv.3"), ("conv.5", "conv.6"),
                       ("conv.8", "conv.9")):
        k = w[f"{conv}.weight"]
        x = _conv64(x, k, w[f"{conv}.bias"], k.shape[-1] // 2)
        x = torch.relu(torch.nn.functional.layer_norm(x, x.shape[1:], w[f"{norm}.weight"],
                                                      w[f"{norm}.bias"]))
    return _heads64(_shared64(x.flatten(1), w), w)


def _fused64(local, rel, glob, w):
    x = torch.relu(_conv64(local.double(), w["l_conv1.weight"], w["l_conv1.bias"], 1))
    x = torch.relu(_conv64(x, w["l_conv2.weight"], w["l_conv2.bias"], 1))
    x = torch.nn.functional.max_pool2d(x, 2).flatten(1)

    def lin(v, k):
        return torch.relu(v @ w[f"{k}.weight"].t() + w[f"{k}.bias"])

    x = lin(x, "l_cnn_fc")
    e = lin(lin(rel.double().flatten(1), "l_rel_fc1"), "l_rel_fc2")
    g = lin(lin(glob.double(), "l_glob_fc1"), "l_glob_fc2")
    return lin(torch.cat([x, e, g], 1), "l_fusion")


def _cell64(x, h, c, w):
    z = (x @ w["lstm.weight_ih_l0"].t() + w["lstm.bias_ih_l0"]
         + h @ w["lstm.weight_hh_l0"].t() + w["lstm.bias_hh_l0"])
    i, f, g, o = z.chunk(4, -1)
    c = torch.sigmoid(f) * c + torch.sigmoid(i) * torch.tanh(g)
    return torch.sigmoid(o) * torch.tanh(c), c


def _ppo64(logits, value, mm, bm, act, old_logp, adv, ret, old_val, cfg, total):
    """The clipped PPO loss of these rows as their share of a batch of `total`,
    and the sums behind the update's statistics."""
    low = torch.finfo(torch.float32).min
    logp, ent = 0.0, 0.0
    for lg, mask, a in ((logits[..., :5], mm, act[..., 0]), (logits[..., 5:7], bm, act[..., 1])):
        ls = torch.log_softmax(lg.masked_fill(~mask.bool(), low), -1)
        logp = logp + ls.gather(-1, a.long().unsqueeze(-1)).squeeze(-1)
        ent = ent - (ls.exp() * ls).sum(-1)
    ratio = torch.exp(logp - old_logp)
    lo, hi = 1 - cfg.clip_eps, 1 + cfg.clip_eps
    pg = -torch.min(ratio * adv, ratio.clamp(lo, hi) * adv).sum() / total
    vc = old_val + (value - old_val).clamp(-cfg.clip_eps, cfg.clip_eps)
    vf = 0.5 * torch.maximum((value - ret).square(), (vc - ret).square()).sum() / total
    en = ent.sum() / total
    stats = torch.stack([pg, vf, en, (old_logp - logp).sum() / total,
                         ((ratio - 1).abs() > cfg.clip_eps).double().sum() / total])
    return pg + cfg.value_coef * vf - cfg.entropy_coef * en, stats.detach()


def exact(case, seed):
    kind = case["kind"]
    if kind in ("step", "tick", "rollout", "versus", "lroll"):
        return None           # a game's rules: compared bit for bit instead
    s = prepare(case, seed)
    w = _f64(s["weights"])
    with torch.no_grad():
        if kind == "act":
            net = _mlp64 if case["net"] == "mlp" else _cnn64
            lg = torch.cat([torch.stack([net(o, w, pid) for pid in range(2)], 1)
                            for o in s["obs"].split(512)])
            return dict(actions=None, logp=None, value=lg[..., 7], logits=lg)
        if kind == "lforward":
            outs = []
            h0, c0 = (x[0].double() for x in s["hidden"])
            for i in range(0, case["n"], 1024):
                x = _fused64(*(f[i:i + 1024] for f in s["feat"]), w)
                h, c = _cell64(x, h0[i:i + 1024], c0[i:i + 1024], w)
                outs.append(torch.cat([_heads64(h, w), h, c], 1))
            o = torch.cat(outs)
            return dict(move=o[:, :5], bomb=o[:, 5:7], value=o[:, 7], h=o[None, :, 8:136],
                        c=o[None, :, 136:])
        if kind == "forward":
            o = torch.cat([_mlp64(x, w, 0) for x in s["obs"].split(65536)])
            return dict(move=o[:, :5], bomb=o[:, 5:7], value=o[:, 7])
    for v in w.values():
        v.requires_grad_(True)
    cfg, stats = s["cfg"], 0.0
    if kind == "grads":
        for r in s["rows"].split(32768):
            o = _mlp64(s["obs"][r], w, 0)
            loss, st = _ppo64(o[:, :7], o[:, 7], s["mm"][r], s["bm"][r], s["act"][r],
                              *(s[k][r].double() for k in ("old_logp", "adv", "ret", "old_val")),
                              cfg, case["rows"])
            loss.backward()
            stats = stats + st
        names = [k for k, _ in s["net"].named_parameters()]
        return dict(stats=stats, grads={k: w[k].grad for k in names})
    # lupdate: advantages over the whole buffer, then the sequences in slices
    buf, n, steps = s["buf"], case["n"], case["steps"]
    rew, val, done = buf.rew.double(), buf.val.double(), buf.done.double()
    adv = torch.empty_like(rew)
    nxt, run_adv = s["last_val"].double(), 0.0
    for t in range(steps - 1, -1, -1):
        live = 1.0 - done[t]
        run_adv = rew[t] + cfg.gamma * nxt * live - val[t] + cfg.gamma * cfg.gae_lambda * live * run_adv
        adv[t], nxt = run_adv, val[t]
    ret = adv + val
    adv = (adv - adv.mean()) / (adv.std() + 1e-8)
    mm, bm, act, lp = buf.mmask, buf.bmask, buf.act, buf.logp.double()
    for i in range(0, n, 128):
        e = slice(i, min(n, i + 128))
        m = e.stop - e.start
        fused = torch.cat([torch.utils.checkpoint.checkpoint(
            lambda a, b, c: _fused64(a, b, c, w), *(x[t:t + 8, e].flatten(0, 1)
                                                    for x in (buf.local, buf.rel, buf.glob)),
            use_reentrant=False) for t in range(0, steps, 8)]).view(steps, m, -1)
        h = c = torch.zeros((m, 128), dtype=torch.float64, device=_dev())
        hs = []
        for t in range(steps):
            h, c = _cell64(fused[t], h, c, w)
            hs.append(h)
            live = (1.0 - done[t, e])[:, None]
            h, c = h * live, c * live
        o = _heads64(torch.stack(hs), w)
        loss, st = _ppo64(o[..., :7], o[..., 7], mm[:, e], bm[:, e], act[:, e], lp[:, e],
                          adv[:, e], ret[:, e], val[:, e], cfg, n * steps)
        loss.backward()
        stats = stats + st
    names = [k for k, _ in s["learner"].named_parameters()]
    norm = torch.stack([w[k].grad.norm() for k in names]).norm()
    scale = (cfg.max_grad_norm / (norm + 1e-6)).clamp(max=1.0)
    order = sorted(("pg", "vf", "ent", "kl", "clipfrac"))
    at = dict(zip(("pg", "vf", "ent", "kl", "clipfrac"), stats))
    return dict(stats=[float(at[k]) for k in order], grads={k: w[k].grad * scale for k in names},
                weights={k: None for k in names if k.startswith("lstm")})
