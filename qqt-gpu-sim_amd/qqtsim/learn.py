"""`HipMlpActorCritic`: the reference's mlp ActorCritic as a trainable module
whose first layer runs forward and backward on the MFMA kernels.

Drop-in for `train/model.py::ActorCritic(arch="mlp")` (:54-259) where the PPO
update uses it (`ppo_update`, train/ppo.py:364-437): same submodules and
state_dict keys (`shared.{0,1,3,4}`, `move_head.{0,2}`, `bomb_head.{0,2}`,
`critic.{0,2}`), `forward(obs, pid)`, `dists`, `evaluate(obs, move_mask,
bomb_mask, actions, pid)`, `n_params`, `arch == "mlp"`, so
`loss.backward()`, `clip_grad_norm_` and the optimizer work unchanged.

The first layer, x (B, 2366) float16 @ W0[:, view columns of pid]^T + b0,
carries nearly all of the update's work and bytes.  Its forward is the
first-layer part of `mlp_act_kernel` (float16 MFMA, W0 rounded to float16
as in acting, float32 accumulation; `qqt_mlp_act` with `z1_out`), its weight
gradient `qqt_l1_grad` (float16 MFMA over the batch, dz1 split hi/lo after
a power-of-two scale, float32 accumulation).  No input gradient is formed
(the observation is data).

Two paths lead through it.  `ppo_grads`, which `ppo_update` takes, runs a
minibatch's loss and everything above the first layer, weight gradients
included, in one kernel (`qqt_ppo_step`).  `forward` / `evaluate` with
autograd keep the reference's own calls: there LayerNorm, the 128-wide layers
and the heads are torch ops (about 8 % of the FLOPs), and their weight
gradients, whose reduction runs over the whole minibatch, batched products over
row chunks (a single batch-long reduction lands on a few workgroups).

`ppo_update` is the reference's update loop (train/ppo.py:364-437) over a
device rollout buffer, with the GAE scan on `qqt_gae`; for the lstm arch
(`LstmLearner`, an lstm rollout buffer) it is the truncated-BPTT update of
train/ppo.py:440-537.
"""

from __future__ import annotations

from dataclasses import dataclass

import torch
from torch import nn

from . import _capi
from .config import n_obs_channels
from .policy import (HEAD, HID, KBLOCK, _layer_tree, column_permutation, default_init, pack_mlp,
                     reference_init)
from .ppo import compute_gae


def _w0_fragments(w: torch.Tensor, cols: torch.Tensor) -> torch.Tensor:
    """(128, k) weight on the device, its columns in the order `cols` ->
    float16 B fragments [tile][kblock][lane][16] (the layout of
    qqtsim.policy._frag), one launch."""
    w = w.detach().float().contiguous()
    n, k = w.shape
    kb = -(-k // KBLOCK)
    out = torch.empty(n * kb * KBLOCK, dtype=torch.float16, device=w.device)
    _capi.check(_capi.lib().qqt_w0_pack(w.data_ptr(), cols.data_ptr(), k, kb, out.data_ptr(),
                                        _capi.stream_handle(w.device)))
    return out


class _FirstLayer(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x16, w0, b0, pid, owner):
        z1 = owner._l1_forward(x16, w0, b0, pid)
        ctx.save_for_backward(x16)
        ctx.pid, ctx.owner = pid, owner
        return z1

    @staticmethod
    def backward(ctx, dz1):
        (x16,) = ctx.saved_tensors
        dw0 = ctx.owner._l1_weight_grad(x16, dz1.contiguous().float(), ctx.pid)
        return None, dw0, dz1.sum(0), None, None


def _weight_grad(dy: torch.Tensor, x: torch.Tensor, chunk: int = 4096) -> torch.Tensor:
    """dy^T x with the batch as the reduction, as batched products over row
    chunks summed in chunk order.  A single product with a batch-long
    reduction runs on a handful of workgroups (the weight is 128 x 128 or
    smaller); chunking spreads it over the GPU."""
    b = dy.shape[0]
    c = b // chunk
    out = None
    if c >= 2:
        n = c * chunk
        dyt = dy[:n].reshape(c, chunk, dy.shape[1]).transpose(1, 2).contiguous()
        out = torch.bmm(dyt, x[:n].reshape(c, chunk, x.shape[1]).contiguous()).sum(0)
        dy, x = dy[n:], x[n:]
    if dy.shape[0]:
        r = dy.t() @ x
        out = r if out is None else out + r
    return out


class _Linear(torch.autograd.Function):
    """F.linear whose weight gradient reduces over the batch in chunks."""

    @staticmethod
    def forward(ctx, x, w, b):
        ctx.save_for_backward(x, w)
        return torch.nn.functional.linear(x, w, b)

    @staticmethod
    def backward(ctx, dy):
        x, w = ctx.saved_tensors
        dy = dy.contiguous()
        return dy @ w, _weight_grad(dy, x), dy.sum(0)


def _seq_weight_grad(dy: torch.Tensor, x: torch.Tensor) -> torch.Tensor:
    """`dy^T x` for the recurrence's weights: chunks short enough that a
    float32 sum within one is no longer than a frame's own product would be
    (error against float64 of dW_ih and dW_hh, 32 frames x 256 envs: chunks of
    256 rows 1.8e-7, of 1,024 2.6e-7, of 4,096 7.4e-7, frame by frame through
    nn.LSTM 2.0e-7; 12 x 37: chunks of 64 6.0e-7, of 256 1.0e-6, nn.LSTM
    6.2e-7), and at most a few hundred of them."""
    rows = dy.shape[0]
    chunk = min(512, max(64, rows // 32))
    c, n = rows // chunk, rows // chunk * chunk
    if c < 2:
        return dy.t() @ x
    out = torch.bmm(dy[:n].reshape(c, chunk, -1).transpose(1, 2),
                    x[:n].reshape(c, chunk, -1)).sum(0)
    return out.addmm_(dy[n:].t(), x[n:]) if n < rows else out


class _InputProduct(_Linear):
    """The same product for the recurrence's inputs, summed over quarters of
    the reduction: one sum over all 256 inputs leaves an error in the gates
    that is larger than everything the recurrence adds (hidden outputs of 32
    frames x 256 envs against float64, mean of eight inputs: 1.37e-7 relative
    with one sum, 1.05e-7 with quarters, 1.06e-7 through nn.LSTM's own
    kernels).  The input gradient sums eighths of its 512 gates: 12 frames x
    37 envs 2.0e-7, in quarters 2.4e-7, through nn.LSTM 1.8e-7."""

    @staticmethod
    def forward(ctx, x, w, b):
        ctx.save_for_backward(x, w)
        step = -(-x.shape[1] // 4)
        parts = [(x[:, k:k + step], w[:, k:k + step].t()) for k in range(0, x.shape[1], step)]
        out = torch.addmm(b, *parts[0])
        for p in parts[1:]:
            out.addmm_(*p)
        return out

    @staticmethod
    def backward(ctx, dy):
        x, w = ctx.saved_tensors
        dy = dy.contiguous()
        eighths = dy.reshape(-1, 8, w.shape[0] // 8).transpose(0, 1)
        dx = torch.bmm(eighths, w.reshape(8, -1, w.shape[1])).sum(0)
        return dx, _seq_weight_grad(dy, x), dy.sum(0)


def _lin(mod: nn.Linear, x):
    return _Linear.apply(x, mod.weight, mod.bias)


class HipMlpActorCritic(nn.Module):
    arch = "mlp"

    def __init__(self, obs_shape=(14, 13, 13), n_moves: int = 5, n_bomb: int = 2,
                 n_players: int = 2, device="cuda", state_dict: dict | None = None):
        super().__init__()
        self.obs_shape = tuple(obs_shape)
        self.n_players = n_players
        if n_obs_channels(n_players) != self.obs_shape[0]:
            raise ValueError("observation channels do not match n_players")
        dev = torch.device(device)
        if dev.type != "cuda":
            raise ValueError("HipMlpActorCritic runs on a ROCm device")
        c, h, w = self.obs_shape
        self.k0 = c * h * w
        self.kpad = -(-self.k0 // KBLOCK) * KBLOCK
        self.shared = nn.Sequential(nn.Linear(self.k0, HID), nn.LayerNorm(HID), nn.ReLU(),
                                    nn.Linear(HID, HID), nn.LayerNorm(HID), nn.ReLU())
        self.move_head = nn.Sequential(nn.Linear(HID, HEAD), nn.ReLU(), nn.Linear(HEAD, n_moves))
        self.bomb_head = nn.Sequential(nn.Linear(HID, HEAD), nn.ReLU(), nn.Linear(HEAD, n_bomb))
        self.critic = nn.Sequential(nn.Linear(HID, HEAD), nn.ReLU(), nn.Linear(HEAD, 1))
        self.load_state_dict(state_dict if state_dict is not None
                             else reference_init(obs_shape, n_moves, n_bomb))
        self.to(dev)
        self._lib = _capi.lib()
        self._perm = [column_permutation(pid, n_players, c, h * w).to(dev)
                      for pid in range(n_players)]
        # the first-layer launch reads the later layers' buffers in its
        # prologue; zero stand-ins of the packed sizes
        packed = pack_mlp(default_init(obs_shape, n_moves, n_bomb), n_players, obs_shape)
        self._stub = {k: torch.zeros_like(v).to(dev) for k, v in packed.items()
                      if torch.is_tensor(v) and k not in ("w0", "b0")}
        self._ws = None

    def n_params(self) -> int:
        return sum(p.numel() for p in self.parameters())

    # ------------------------------------------------------------ kernels
    @staticmethod
    def _rows_args(a, x16, rows):
        """Batch = x16's rows, or, with `rows` (int64 indices into x16),
        those rows read in place."""
        if rows is None:
            return x16.shape[0]
        if rows.dtype != torch.int64 or not rows.is_contiguous() or rows.device != x16.device:
            raise ValueError("rows must be a contiguous int64 tensor on the observation's device")
        a.row_index, a.obs_rows = rows.data_ptr(), x16.shape[0]
        return rows.numel()

    def _l1_forward(self, x16, w0, b0, pid, rows=None):
        a = _capi.MlpArgsC()
        b = self._rows_args(a, x16, rows)
        z1 = torch.empty((b, HID), dtype=torch.float32, device=x16.device)
        frag = _w0_fragments(w0, self._perm[pid])
        bias = b0.detach().float().contiguous()
        a.batch, a.npid, a.pid0, a.sample = b, 1, 0, 0
        a.k0, a.kblocks0, a.obs_stride = self.k0, self.kpad // KBLOCK, x16.stride(0)
        a.w0_players = 1
        a.obs, a.w0, a.b0 = x16.data_ptr(), frag.data_ptr(), bias.data_ptr()
        for k, v in self._stub.items():
            setattr(a, k, v.data_ptr())
        a.z1_out = z1.data_ptr()
        _capi.check(self._lib.qqt_mlp_act(a, _capi.stream_handle(x16.device)))
        return z1

    def _l1_weight_grad(self, x16, dz1, pid, scale=None, rows=None):
        """dW0 of the rows of x16 (or of its rows `rows`) against dz1; `scale`
        (device, 1 value) = the power of two that brings max |dz1| to ~2^14
        when the caller has it."""
        a = _capi.L1GradArgsC()
        b = self._rows_args(a, x16, rows)
        need = int(self._lib.qqt_l1_grad_preferred_floats(b, self.k0))
        if self._ws is None or self._ws.numel() < need:
            self._ws = torch.empty(need, dtype=torch.float32, device=x16.device)
        if scale is None:
            amax = dz1.abs().amax().clamp_min(1e-30)
            scale = torch.exp2(torch.clamp(14.0 - torch.ceil(torch.log2(amax)), -100.0, 100.0))
        dw0 = torch.empty((HID, self.k0), dtype=torch.float32, device=x16.device)
        a.batch, a.k0, a.obs_stride = b, self.k0, x16.stride(0)
        a.workspace_floats = self._ws.numel()
        a.obs, a.dz1, a.dz_scale = x16.data_ptr(), dz1.data_ptr(), scale.data_ptr()
        a.workspace, a.dw0 = self._ws.data_ptr(), dw0.data_ptr()
        _capi.check(self._lib.qqt_l1_grad_columns(a, self._perm[pid].data_ptr(),
                                                  _capi.stream_handle(x16.device)))
        return dw0

    # ------------------------------------------------------------ API
    def forward(self, obs, pid: int = 0):
        """(move logits, bomb logits, value) like train/model.py:167-196."""
        b = obs.shape[0]
        x16 = obs.reshape(b, -1)
        if x16.dtype != torch.float16:
            x16 = x16.half()
        x16 = x16.contiguous()
        if x16.shape[1] != self.k0:
            raise ValueError(f"observation rows must have {self.k0} values")
        lin = self.shared[0]
        x = _FirstLayer.apply(x16, lin.weight, lin.bias, int(pid), self)
        x = torch.relu(self.shared[1](x))
        x = torch.relu(self.shared[4](_lin(self.shared[3], x)))
        heads = [_lin(h[2], torch.relu(_lin(h[0], x)))
                 for h in (self.move_head, self.bomb_head, self.critic)]
        return heads[0], heads[1], heads[2].squeeze(-1)

    @staticmethod
    def masked_dist(logits, mask):
        neg_inf = torch.finfo(logits.dtype).min
        masked = torch.where(mask, logits, torch.full_like(logits, neg_inf))
        return torch.distributions.Categorical(logits=masked)

    def dists(self, obs, move_mask, bomb_mask, pid: int = 0):
        ml, bl, val = self(obs, pid)
        return (self.masked_dist(ml, move_mask.bool()), self.masked_dist(bl, bomb_mask.bool()),
                val)

    def ppo_grads(self, obs, move_mask, bomb_mask, actions, old_logp, adv, ret, old_val,
                  cfg, entropy_coef: float, rows=None) -> torch.Tensor:
        """Gradients of the reference's minibatch PPO loss (train/ppo.py:401-421,
        player 0's view) written into every parameter's `.grad`, as
        `loss.backward()` through `evaluate` would leave them; returns the
        five statistics (pg, vf, ent, kl, clipfrac) as a device tensor.
        Four calls: the first layer's weight fragments and forward,
        `qqt_ppo_step` (the loss, the backward above the first layer and every
        gradient there) and `qqt_l1_grad_columns`.  With `rows` (int64 indices), every per-row argument (obs,
        masks, actions, old log-probs, advantages, returns, old values) is a
        whole buffer and the minibatch is its rows `rows`, which the kernels
        read in place."""
        dev = obs.device
        x16 = obs.reshape(obs.shape[0], -1)
        x16 = (x16 if x16.dtype == torch.float16 else x16.half()).contiguous()
        b = x16.shape[0] if rows is None else rows.numel()
        l0, ln1, l1, ln2 = (self.shared[i] for i in (0, 1, 3, 4))
        heads = (self.move_head, self.bomb_head, self.critic)
        if [h[2].weight.shape[0] for h in heads] != [5, 2, 1]:
            raise ValueError("ppo_grads serves heads of 5 moves, 2 bomb actions and the value")
        if rows is not None and any(t.shape[0] != x16.shape[0] for t in (
                move_mask, bomb_mask, actions, old_logp, adv, ret, old_val)):
            raise ValueError("with rows, every per-row argument must be a whole buffer")
        z1 = self._l1_forward(x16, l0.weight, l0.bias, 0, rows)
        a = _capi.PpoStepArgsC()
        keep, grads = [], []

        def put(name, t, slot=None):
            keep.append(t)
            if slot is None:
                setattr(a, name, t.data_ptr())
            else:
                getattr(a, name)[slot] = t.data_ptr()

        def param(name, p, slot=None):      # the parameter itself and its new gradient
            t = p.detach().float().contiguous()
            # a parameter that is a view into a flat buffer may lie at any element
            put(name, t.clone() if t.data_ptr() % 16 else t, slot)
            grads.append((p, torch.empty(p.shape, dtype=torch.float32, device=dev)))
            put("d" + name, grads[-1][1], slot)

        for name, p in (("ln1_w", ln1.weight), ("ln1_b", ln1.bias), ("w1", l1.weight),
                        ("b1", l1.bias), ("ln2_w", ln2.weight), ("ln2_b", ln2.bias)):
            param(name, p)
        for i, h in enumerate(heads):
            for name, p in (("wh", h[0].weight), ("bh", h[0].bias), ("wf", h[2].weight),
                            ("bf", h[2].bias)):
                param(name, p, i)
        if rows is not None:
            a.row_index, a.src_rows = rows.data_ptr(), x16.shape[0]
        f32 = dict(dtype=torch.float32, device=dev)
        dz1, scale, stats, db0 = (torch.empty(s, **f32) for s in ((b, HID), (1,), (5,), (HID,)))
        need = int(self._lib.qqt_ppo_step_workspace_bytes(b))
        for name, t in (("z1", z1), ("actions", actions.to(torch.int64).contiguous()),
                        ("move_mask", move_mask.to(torch.uint8).contiguous()),
                        ("bomb_mask", bomb_mask.to(torch.uint8).contiguous()),
                        ("old_logp", old_logp.float().contiguous()), ("adv", adv.float().contiguous()),
                        ("ret", ret.float().contiguous()), ("old_val", old_val.float().contiguous()),
                        ("dz1", dz1), ("dz_scale", scale), ("stats", stats), ("db0", db0),
                        ("workspace", torch.empty((need,), dtype=torch.uint8, device=dev))):
            put(name, t)
        a.batch, a.workspace_bytes = b, need
        a.clip_eps = cfg.clip_eps
        a.ratio_lo, a.ratio_hi = 1 - cfg.clip_eps, 1 + cfg.clip_eps
        a.value_coef, a.entropy_coef = cfg.value_coef, entropy_coef
        _capi.check(self._lib.qqt_ppo_step(a, _capi.stream_handle(dev)))
        grads += [(l0.bias, db0), (l0.weight, self._l1_weight_grad(x16, dz1, 0, scale=scale, rows=rows))]
        for p, g in grads:      # only now: a call that is refused leaves every `.grad` as it was
            p.grad = g
        return stats

    def evaluate(self, obs, move_mask, bomb_mask, actions, pid: int = 0):
        """(logp, entropy, value) of given actions (train/model.py:247-256)."""
        dm, db, val = self.dists(obs, move_mask, bomb_mask, pid)
        logp = dm.log_prob(actions[..., 0]) + db.log_prob(actions[..., 1])
        return logp, dm.entropy() + db.entropy(), val


@dataclass
class PPOConfig:
    """train/ppo.py:38-51."""
    rollout_steps: int = 128
    epochs: int = 4
    minibatches: int = 4
    gamma: float = 0.995
    gae_lambda: float = 0.95
    clip_eps: float = 0.2
    value_coef: float = 0.5
    entropy_coef: float = 0.05
    entropy_final: float = 0.03
    max_grad_norm: float = 0.5
    lr: float = 3e-4
    oversample_dying: int = 3
    bptt_window: int = 0


def _gather_rows(x: torch.Tensor, sel: torch.Tensor) -> torch.Tensor:
    """x[sel] for a contiguous device tensor whose rows are whole 4-byte
    words (the observation rows: 2366 float16), as one `qqt_gather_rows`
    launch (~1.6x torch's row gather of the same bytes); other tensors go
    through torch indexing."""
    n = x.shape[0]
    row_bytes = x[0].numel() * x.element_size() if n else 0
    if not (x.is_cuda and x.is_contiguous() and row_bytes % 4 == 0 and row_bytes > 0):
        return x[sel]
    idx = sel.to(torch.int64).contiguous()
    out = torch.empty((idx.numel(),) + tuple(x.shape[1:]), dtype=x.dtype, device=x.device)
    a = _capi.GatherArgsC()
    a.n, a.row_words = idx.numel(), row_bytes // 4
    a.src_rows, a.src_stride, a.dst_stride = n, row_bytes // 4, row_bytes // 4
    a.src, a.dst, a.index = x.data_ptr(), out.data_ptr(), idx.data_ptr()
    _capi.check(_capi.lib().qqt_gather_rows(a, _capi.stream_handle(x.device)))
    return out


class _Transitions:
    """A filled buffer's learner transitions as flat (T*N, ...) rows: the
    observation, masks, actions, the log-probabilities and values the
    acting network recorded, and the GAE targets (advantages normalised
    over the whole buffer with the unbiased standard deviation + 1e-8,
    train/ppo.py:374)."""

    FIELDS = ("obs", "mmask", "bmask", "act", "old_logp", "adv", "ret", "old_val")

    def __init__(self, buf, adv: torch.Tensor, ret: torch.Tensor):
        def rows(x):
            return x.reshape(x.shape[0] * x.shape[1], *x.shape[2:])
        self.obs, self.mmask, self.bmask = rows(buf.obs), rows(buf.mmask), rows(buf.bmask)
        self.act, self.old_logp, self.old_val = rows(buf.act), rows(buf.logp), rows(buf.val)
        a = rows(adv)
        self.adv = (a - a.mean()) / (a.std() + 1e-8)
        self.ret = rows(ret)
        self.count = self.obs.shape[0]

    def select(self, idx: torch.Tensor) -> dict:
        """The rows `idx` of every field (the observation by `qqt_gather_rows`)."""
        out = {k: getattr(self, k)[idx] for k in self.FIELDS if k != "obs"}
        out["obs"] = _gather_rows(self.obs, idx)
        return out


def _draw_pool(buf, count: int, repeats: int, device) -> torch.Tensor:
    """Row indices the epochs draw from (train/ppo.py:381-394): every row
    once, followed by the rows where player 0 took damage or the episode
    ended repeated `repeats - 1` more times (in row order), when there are
    any and `repeats > 1`."""
    every = torch.arange(count, device=device)
    if repeats <= 1:
        return every
    hurt_or_done = buf.dmg.reshape(count) | buf.done.reshape(count).bool()
    rare = hurt_or_done.nonzero(as_tuple=False).squeeze(1)
    if rare.numel() == 0:
        return every
    return torch.cat([every, rare.repeat(repeats - 1)])


def _minibatch_plan(pool: torch.Tensor, count: int, epochs: int, minibatches: int):
    """Yields each minibatch's row indices: per epoch, one `randperm` over
    the pool (the default generator of the pool's device), its first `count`
    entries cut into consecutive slices of `max(1, count // minibatches)`
    (a shorter last slice when that does not divide `count`),
    train/ppo.py:395-405."""
    size = max(1, count // minibatches)
    for _ in range(epochs):
        order = pool[torch.randperm(pool.numel(), device=pool.device)][:count]
        for lo in range(0, count, size):
            yield order[lo:lo + size]


def _autograd_minibatch(learner, mb: dict, cfg, entropy_coef: float):
    """The reference's minibatch loss (train/ppo.py:406-421) through the
    learner's `evaluate` and autograd; returns the loss and the five
    statistics (pg, vf, ent, kl, clipfrac) as a device tensor."""
    logp, ent, value = learner.evaluate(mb["obs"], mb["mmask"], mb["bmask"], mb["act"])
    adv, old_val, ret = mb["adv"], mb["old_val"], mb["ret"]
    ratio = torch.exp(logp - mb["old_logp"])
    surrogate = torch.min(ratio * adv, torch.clamp(ratio, 1 - cfg.clip_eps, 1 + cfg.clip_eps) * adv)
    pg = -surrogate.mean()
    value_clipped = old_val + torch.clamp(value - old_val, -cfg.clip_eps, cfg.clip_eps)
    vf = 0.5 * torch.maximum((value - ret).square(), (value_clipped - ret).square()).mean()
    ent_mean = ent.mean()
    loss = pg + cfg.value_coef * vf - entropy_coef * ent_mean
    with torch.no_grad():
        stats = torch.stack([pg, vf, ent_mean, (mb["old_logp"] - logp).mean(),
                             ((ratio - 1).abs() > cfg.clip_eps).float().mean()])
    return loss, stats


UPDATE_STATS = ("pg", "vf", "ent", "kl", "clipfrac")


class LstmLearner(nn.Module):
    """The reference's lstm ActorCritic (train/model.py:103-120, 148-153,
    176-214, 247-256) as a trainable torch module: the same submodules and
    state_dict keys (`l_conv1` .. `l_fusion`, `lstm`, the heads), so its
    weights load into `HipLstmActorCritic` for acting and back.  It computes
    with torch ops (convolutions, the LSTM and the products run on the
    device's libraries) and serves the lstm PPO update."""

    arch = "lstm"

    def __init__(self, obs_shape=(14, 13, 13), n_moves: int = 5, n_bomb: int = 2,
                 state_dict: dict | None = None, seed: int = 0):
        super().__init__()
        tree = _layer_tree("lstm", tuple(obs_shape), n_moves, n_bomb)
        for name, mod in tree.named_children():
            self.add_module(name, mod)
        self.l_pool = nn.MaxPool2d(2)
        self.obs_shape = tuple(obs_shape)
        self.load_state_dict(state_dict if state_dict is not None
                             else reference_init(obs_shape, n_moves, n_bomb, seed, arch="lstm"))

    def n_params(self) -> int:
        return sum(p.numel() for p in self.parameters())

    def extract_fused(self, local, rel, glob):
        """(B, 256) fused per-frame features (train/model.py:198-214)."""
        r = torch.relu
        w = self.l_conv1.weight
        x = self.l_pool(r(self.l_conv2(r(self.l_conv1(local.to(w.dtype))))))
        x = r(self.l_cnn_fc(x.flatten(1)))
        e = r(self.l_rel_fc2(r(self.l_rel_fc1(rel.to(w.dtype).flatten(1)))))
        g = r(self.l_glob_fc2(r(self.l_glob_fc1(glob.to(w.dtype)))))
        return r(self.l_fusion(torch.cat([x, e, g], 1)))

    def heads(self, h):
        return self.move_head(h), self.bomb_head(h), self.critic(h).squeeze(-1)

    def forward(self, obs, pid: int = 0, hidden=None):
        """(move logits, bomb logits, value, hidden') of one frame; `obs` =
        (local, rel, glob), `hidden` = ((1,B,128), (1,B,128)) or None."""
        out, nh = self.lstm(self.extract_fused(*obs).unsqueeze(1), hidden)
        return (*self.heads(out.squeeze(1)), nh)

    def evaluate(self, obs, move_mask, bomb_mask, actions, pid: int = 0, hidden=None):
        ml, bl, v, _ = self(obs, pid, hidden)
        logp, ent = _masked_logp_entropy(ml, bl, move_mask, bomb_mask, actions)
        return logp, ent, v


def _masked_logp_entropy(ml, bl, mm, bm, act):
    """log-probability of `act` and entropy of the factored masked
    distribution: the reference's Categorical over logits with the masked
    entries set to the dtype's lowest value (train/model.py:215-220)."""
    logp, ent = 0.0, 0.0
    for logits, mask, a in ((ml, mm, act[..., 0]), (bl, bm, act[..., 1])):
        low = torch.finfo(logits.dtype).min
        ls = torch.log_softmax(torch.where(mask.bool(), logits, torch.full_like(logits, low)), -1)
        logp = logp + ls.gather(-1, a.long().unsqueeze(-1)).squeeze(-1)
        ent = ent - (ls.exp() * ls).sum(-1)
    return logp, ent


def _aligned(t: torch.Tensor) -> torch.Tensor:
    """t, contiguous and on 16 bytes (a view into a flat buffer, a parameter or
    one that a saved-tensor hook returns, may lie at any element)."""
    t = t.contiguous()
    return t.clone() if t.data_ptr() % 16 else t


class _Recurrence(torch.autograd.Function):
    """(T, m, 128) hidden outputs of the recurrence z = zx + h W_hh^T over T
    frames from the zero state, the state multiplied by keep[t] after frame t
    and detached every `window` frames (0 = never): one launch forward, one
    backward (`qqt_lstm_seq_*`).  W_hh's gradient is one product over all
    frames after the first."""

    @staticmethod
    def forward(ctx, zx, w_hh, keep, window):
        steps, m = keep.shape
        new = lambda width: torch.empty((steps, m, width), dtype=torch.float32,  # noqa: E731
                                        device=zx.device)
        h, c, gates = new(HID), new(HID), new(4 * HID)
        a = _capi.LstmSeqArgsC()
        a.steps, a.rows, a.window = steps, m, window
        a.w_hh, a.keep, a.zx = w_hh.data_ptr(), keep.data_ptr(), zx.data_ptr()
        a.h, a.c, a.gates = h.data_ptr(), c.data_ptr(), gates.data_ptr()
        _capi.check(_capi.lib().qqt_lstm_seq_forward(a, _capi.stream_handle(zx.device)))
        ctx.save_for_backward(w_hh, keep, h, c, gates)
        ctx.window = window
        return h

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, dh):
        w_hh, keep, h, c, gates = ctx.saved_tensors
        w_hh = _aligned(w_hh)
        keep, h, c, gates, dh = (t.contiguous() for t in (keep, h, c, gates, dh))
        dz = torch.empty_like(gates)
        a = _capi.LstmSeqArgsC()
        a.steps, a.rows, a.window = *keep.shape, ctx.window
        a.w_hh, a.keep, a.c, a.gates = (t.data_ptr() for t in (w_hh, keep, c, gates))
        a.dh, a.dz = dh.data_ptr(), dz.data_ptr()
        _capi.check(_capi.lib().qqt_lstm_seq_backward(a, _capi.stream_handle(dh.device)))
        dw = None
        if ctx.needs_input_grad[1]:
            if keep.shape[0] > 1:
                before = (h[:-1] * keep[:-1].unsqueeze(-1)).view(-1, HID)
                dw = _seq_weight_grad(dz[1:].view(-1, 4 * HID), before)
            else:
                dw = torch.zeros_like(w_hh)
        return dz if ctx.needs_input_grad[0] else None, dw, None, None


def _sequence_kernels_serve(lstm, x) -> bool:
    """Whether `_Recurrence` stands for the module's own call frame by frame:
    a plain float32 nn.LSTM of this network's shape on the GPU, with nothing
    hooked into its call or its parameters' use."""
    if type(lstm) is not nn.LSTM or not x.is_cuda or x.dtype != torch.float32:
        return False
    if (lstm.num_layers, lstm.hidden_size, lstm.bidirectional, lstm.proj_size, lstm.bias,
            lstm.batch_first) != (1, HID, False, 0, True, True):
        return False
    if "forward" in vars(lstm) or any(getattr(lstm, k, None) for k in (
            "_forward_hooks", "_forward_pre_hooks", "_backward_hooks", "_backward_pre_hooks")):
        return False
    mod = torch.nn.modules.module
    if any(getattr(mod, k, None) for k in ("_global_forward_hooks", "_global_forward_pre_hooks",
                                           "_global_backward_hooks",
                                           "_global_backward_pre_hooks")):
        return False
    if torch.is_autocast_enabled() or torch.compiler.is_compiling():
        return False
    w = (lstm.weight_ih_l0, lstm.weight_hh_l0, lstm.bias_ih_l0, lstm.bias_hh_l0)
    return all(p.dtype == torch.float32 and p.device == x.device for p in w)


def _sequence_outputs(lstm, fused, keep, window: int):
    """(T, m, 128) outputs of the LSTM over the fused features (T, m, 256):
    the input products of all frames together, then the recurrence."""
    steps, m, width = fused.shape
    zx = _InputProduct.apply(fused.reshape(steps * m, width), lstm.weight_ih_l0,
                       lstm.bias_ih_l0 + lstm.bias_hh_l0)
    return _Recurrence.apply(zx.view(steps, m, -1).contiguous(), _aligned(lstm.weight_hh_l0),
                             keep.contiguous(), window)


def _lstm_update(learner, opt, buf, last_val, cfg: PPOConfig, entropy_coef: float) -> dict:
    """PPO over an lstm rollout buffer (train/ppo.py:440-537).  Minibatches
    are sets of envs with their whole T-step sequences: per epoch one
    `randperm` over the N envs (the default generator of the buffer's
    device) cut into slices of max(1, N // minibatches).  Per minibatch the
    per-frame features of all T x N_sub frames go through `extract_fused`
    at once; the LSTM then runs over t = 0..T-1 from the zero state, its
    state multiplied by (1 - done[t]) after each frame and detached every
    `bptt_window` frames (0 = never), as one forward and one backward launch
    where `_sequence_kernels_serve` says so (frame by frame through the module
    it is about 1,500 launches per minibatch of 32 frames); the heads and the masked log-probs
    run on all frames together.  The clipped surrogate, the clipped value
    loss and the entropy bonus use the GAE advantages normalised over the
    whole buffer (unbiased std + 1e-8); then gradient clipping and one
    optimizer step.  Returns the mean statistics over minibatches."""
    adv, ret = compute_gae(buf, last_val, cfg.gamma, cfg.gae_lambda)
    adv = (adv - adv.mean()) / (adv.std() + 1e-8)
    steps, n = adv.shape
    dev = adv.device
    size = max(1, n // cfg.minibatches)
    keep = 1.0 - buf.done                                   # (T, N) float32
    old_logp, old_val = buf.logp, buf.val
    mm, bm, act = buf.mmask, buf.bmask, buf.act
    window = int(getattr(cfg, "bptt_window", 0))
    params = list(learner.parameters())
    total = torch.zeros(len(UPDATE_STATS), dtype=torch.float32, device=dev)
    count = 0
    for _ in range(cfg.epochs):
        order = torch.randperm(n, device=dev)
        for lo in range(0, n, size):
            envs = order[lo:lo + size]
            m = envs.numel()
            frames = [x[:, envs].reshape(steps * m, *x.shape[2:])
                      for x in (buf.local, buf.rel, buf.glob)]
            fused = learner.extract_fused(*frames).view(steps, m, -1)
            if steps > 0 and _sequence_kernels_serve(learner.lstm, fused):
                hidden = _sequence_outputs(learner.lstm, fused, keep[:, envs], max(0, window))
            else:
                k = keep[:, envs].view(steps, 1, m, 1)
                state, outs = None, []
                for t in range(steps):
                    if window > 0 and t % window == 0 and state is not None:
                        state = (state[0].detach(), state[1].detach())
                    out, state = learner.lstm(fused[t].unsqueeze(1), state)
                    outs.append(out.squeeze(1))
                    state = (state[0] * k[t], state[1] * k[t])
                hidden = torch.stack(outs)
            ml, bl, value = learner.heads(hidden)
            logp, ent = _masked_logp_entropy(ml, bl, mm[:, envs], bm[:, envs], act[:, envs])
            a, r, ov, ol = adv[:, envs], ret[:, envs], old_val[:, envs], old_logp[:, envs]
            ratio = torch.exp(logp - ol)
            pg = -torch.min(ratio * a, torch.clamp(ratio, 1 - cfg.clip_eps, 1 + cfg.clip_eps) * a
                            ).mean()
            vc = ov + torch.clamp(value - ov, -cfg.clip_eps, cfg.clip_eps)
            vf = 0.5 * torch.maximum((value - r).square(), (vc - r).square()).mean()
            ent_mean = ent.mean()
            loss = pg + cfg.value_coef * vf - entropy_coef * ent_mean
            opt.zero_grad(set_to_none=True)
            loss.backward()
            torch.nn.utils.clip_grad_norm_(params, cfg.max_grad_norm)
            opt.step()
            with torch.no_grad():
                total += torch.stack([pg, vf, ent_mean, (ol - logp).mean(),
                                      ((ratio - 1).abs() > cfg.clip_eps).float().mean()])
            count += 1
    return dict(zip(UPDATE_STATS, (total / max(1, count)).tolist()))


def ppo_update(learner, opt, buf, last_val, cfg: PPOConfig, entropy_coef: float) -> dict:
    """One PPO update over a filled rollout buffer (train/ppo.py:364-437).

    GAE runs as one `qqt_gae` launch.  Each minibatch's gradients come from
    the learner's fused loss + backward (`ppo_grads`, HipMlpActorCritic) or,
    for any other learner, from autograd through `evaluate`; then gradient
    clipping to `max_grad_norm` and one optimizer step.  The statistics
    stay on the device until the end and are returned as the mean over
    minibatches, like the reference's dict.  An lstm buffer (or learner)
    takes the truncated-BPTT update of `_lstm_update`."""
    if getattr(buf, "arch", None) == "lstm" or getattr(learner, "arch", None) == "lstm":
        if getattr(buf, "arch", None) != "lstm" or getattr(learner, "arch", None) != "lstm":
            raise ValueError("the lstm update needs an lstm learner and an lstm rollout buffer")
        return _lstm_update(learner, opt, buf, last_val, cfg, entropy_coef)
    adv, ret = compute_gae(buf, last_val, cfg.gamma, cfg.gae_lambda)
    data = _Transitions(buf, adv, ret)
    dev = data.obs.device
    pool = _draw_pool(buf, data.count, cfg.oversample_dying, dev)
    fused = getattr(learner, "ppo_grads", None)
    params = list(learner.parameters())
    total = torch.zeros(len(UPDATE_STATS), dtype=torch.float32, device=dev)
    steps = 0
    if fused is not None:          # its kernels read every minibatch row in place
        whole = dict(mm=data.mmask.to(torch.uint8).contiguous(),
                     bm=data.bmask.to(torch.uint8).contiguous(),
                     act=data.act.to(torch.int64).contiguous(),
                     **{k: getattr(data, k).float().contiguous()
                        for k in ("old_logp", "adv", "ret", "old_val")})
    for idx in _minibatch_plan(pool, data.count, cfg.epochs, cfg.minibatches):
        opt.zero_grad(set_to_none=True)
        if fused is not None:
            stats = fused(data.obs, whole["mm"], whole["bm"], whole["act"], whole["old_logp"],
                          whole["adv"], whole["ret"], whole["old_val"], cfg, entropy_coef,
                          rows=idx.contiguous())
        else:
            mb = data.select(idx)
            loss, stats = _autograd_minibatch(learner, mb, cfg, entropy_coef)
            loss.backward()
        torch.nn.utils.clip_grad_norm_(params, cfg.max_grad_norm)
        opt.step()
        total += stats
        steps += 1
    return dict(zip(UPDATE_STATS, (total / max(1, steps)).tolist()))
