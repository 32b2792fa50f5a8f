"""qqt_ppo_step (the fused PPO minibatch with in-kernel weight gradients)
against float64 torch from the same first-layer output (needs an MI355X),
and its argument checks (no GPU needed)."""

import ctypes

import pytest
import torch

K0 = 14 * 13 * 13


def _case(b, seed, dev, outliers):
    g = torch.Generator().manual_seed(seed)
    obs = (torch.rand((b, K0), generator=g) < 0.2).half().to(dev)
    mm = (torch.rand((b, 5), generator=g) < 0.6).to(dev)
    mm[:, 4] = True
    bm = torch.ones((b, 2), dtype=torch.bool, device=dev)
    bm[:, 1] = (torch.rand(b, generator=g) < 0.5).to(dev)
    act = torch.stack([torch.multinomial(mm.float().cpu(), 1, generator=g)[:, 0],
                       torch.multinomial(bm.float().cpu(), 1, generator=g)[:, 0]], 1).to(dev)
    f = lambda s: (s * torch.randn(b, generator=g)).to(dev)  # noqa: E731
    old_logp, adv, ret, old_val = f(0.3) - 1.5, f(1.0), f(1.0), f(1.0)
    if outliers:                 # rows whose gradients are orders of magnitude above the others'
        adv[b // 2], ret[-1] = 3e4, 1e5
    return obs, mm, bm, act, old_logp, adv, ret, old_val


def _float64(net, z1, mm, bm, act, old_logp, adv, ret, old_val, cfg):
    """Gradients of the minibatch loss above layer 1 (train/ppo.py:408-421)."""
    w = {k: v.detach().double().requires_grad_(True) for k, v in net.named_parameters()
         if k != "shared.0.weight"}
    ln = torch.nn.functional.layer_norm
    x = z1.double() + (w["shared.0.bias"] - w["shared.0.bias"].detach())
    x = torch.relu(ln(x, (128,), w["shared.1.weight"], w["shared.1.bias"]))
    x = x @ w["shared.3.weight"].t() + w["shared.3.bias"]
    x = torch.relu(ln(x, (128,), w["shared.4.weight"], w["shared.4.bias"]))
    o = []
    for h in ("move_head", "bomb_head", "critic"):
        y = torch.relu(x @ w[f"{h}.0.weight"].t() + w[f"{h}.0.bias"])
        o.append(y @ w[f"{h}.2.weight"].t() + w[f"{h}.2.bias"])
    logp, ent = 0.0, 0.0
    for lg, mask, a in ((o[0], mm, act[:, 0]), (o[1], bm, act[:, 1])):
        ls = torch.log_softmax(lg.masked_fill(~mask, torch.finfo(torch.float32).min), -1)
        logp = logp + ls.gather(-1, a[:, None])[:, 0]
        ent = ent - (ls.exp() * ls).sum(-1)
    v, e = o[2][:, 0], cfg.clip_eps
    ratio = (logp - old_logp.double()).exp()
    pg = -torch.min(ratio * adv, ratio.clamp(1 - e, 1 + e) * adv).mean()
    vc = old_val + (v - old_val).clamp(-e, e)
    vf = 0.5 * torch.maximum((v - ret) ** 2, (vc - ret) ** 2).mean()
    (pg + cfg.value_coef * vf - 0.05 * ent.mean()).backward()
    return {k: p.grad for k, p in w.items()}, torch.stack([pg, vf, ent.mean()]).detach()


@pytest.mark.gpu
@pytest.mark.parametrize("outliers", [False, True])
@pytest.mark.parametrize("b", [1, 31, 32, 33, 100, 8193])
def test_gradients_against_float64(b, outliers):
    """Batches around the 32-row tile, one past a whole round of the 256
    workgroups, and a batch whose gradients span nine orders of magnitude.
    Bound: float32 products of 128 and 192 terms through four layers are
    within 3e-6 relative; a hidden unit within rounding of zero may pass or
    block its ReLU gradient, one row's share of the sum, so 2e-4 beyond a few
    rows (the outlier row carries its whole sum)."""
    from qqtsim import HipMlpActorCritic, PPOConfig, reference_init

    dev = torch.device("cuda:0")
    sd = reference_init(seed=b)
    for k in sd:
        if k.endswith("2.weight"):
            sd[k] = sd[k] + 0.1 * torch.randn(sd[k].shape, generator=torch.Generator().manual_seed(1))
    net = HipMlpActorCritic(device=dev, state_dict=sd)
    cfg = PPOConfig()
    args = _case(b, b, dev, outliers)
    z1 = net._l1_forward(args[0], net.shared[0].weight, net.shared[0].bias, 0)
    want, want_st = _float64(net, z1, *args[1:], cfg)
    st = net.ppo_grads(*args, cfg, 0.05)
    for k, p in net.named_parameters():
        if k in want:
            scale = want[k].norm()
            err = float((p.grad.double() - want[k]).norm())
            assert err <= (2e-4 if b > 32 else 3e-6) * float(scale) + 1e-12, (k, err / float(scale))
    assert float(((st[:3] - want_st) / want_st.abs().clamp_min(1.0)).abs().max()) <= 1e-5
    dw0 = net.shared[0].weight.grad
    assert bool(torch.isfinite(dw0).all()) and float(dw0.abs().max()) > 0.0


def _row_losses(w, z1, mm, bm, act, old_logp, adv, ret, old_val, cfg, entropy_coef):
    """Each row's loss in float64 and how far it is from the nearest kink (a
    ReLU input at zero, a ratio or value at its clip bound, a tie of the two
    value errors)."""
    ln = torch.nn.functional.layer_norm
    a1 = ln(z1, (128,), w["shared.1.weight"], w["shared.1.bias"])
    a2 = ln(torch.relu(a1) @ w["shared.3.weight"].t() + w["shared.3.bias"], (128,),
            w["shared.4.weight"], w["shared.4.bias"])
    near, o = [a1, a2], []
    for h in ("move_head", "bomb_head", "critic"):
        near.append(torch.relu(a2) @ w[f"{h}.0.weight"].t() + w[f"{h}.0.bias"])
        o.append(torch.relu(near[-1]) @ w[f"{h}.2.weight"].t() + w[f"{h}.2.bias"])
    logp, ent = 0.0, 0.0
    for lg, mask, a in ((o[0], mm, act[:, 0]), (o[1], bm, act[:, 1])):
        ls = torch.log_softmax(lg.masked_fill(~mask, torch.finfo(torch.float32).min), -1)
        logp = logp + ls.gather(-1, a[:, None])[:, 0]
        ent = ent - (ls.exp() * ls).sum(-1)
    v, e = o[2][:, 0], cfg.clip_eps
    ratio, dv = (logp - old_logp.double()).exp(), v - old_val
    vc = old_val + dv.clamp(-e, e)
    loss = (-torch.min(ratio * adv, ratio.clamp(1 - e, 1 + e) * adv) - entropy_coef * ent
            + 0.5 * cfg.value_coef * torch.maximum((v - ret) ** 2, (vc - ret) ** 2))
    tie = torch.where(vc == v, torch.ones_like(v), ((v - ret).abs() - (vc - ret).abs()).abs())
    near = [torch.cat(near, 1).abs().amin(1), (ratio - 1 - e).abs(), (ratio - 1 + e).abs(),
            (dv.abs() - e).abs(), tie]
    return loss, torch.stack(near).amin(0)


def _smooth_rows(net, b, seed, dev, cfg, entropy_coef, scale_rows):
    """b rows of `_case` none of which is within rounding of a kink (there a
    correct float32 result may take either branch), their z1 and weights."""
    args = _case(b + b // 8 + 64, seed, dev, False)
    old_logp, adv, ret, old_val = args[4:]
    scale_rows(adv, ret, old_val)
    lin = net.shared[0]
    w = {k: v.detach().double() for k, v in net.named_parameters()}
    with torch.no_grad():
        z1 = net._l1_forward(args[0], lin.weight, lin.bias, 0)
        near = _row_losses(w, z1.double(), *args[1:], cfg, entropy_coef)[1]
        keep = (near > 3e-6).nonzero()[:, 0][:b]
        assert keep.numel() == b
        args = tuple(x[keep].contiguous() for x in args)
        return args, net._l1_forward(args[0], lin.weight, lin.bias, 0), w


def _spread_net(seed, dev):
    from qqtsim import HipMlpActorCritic, reference_init

    sd = reference_init(seed=seed)
    g = torch.Generator().manual_seed(seed)
    for k in sd:
        if k.endswith("2.weight"):
            sd[k] = sd[k] + 0.1 * torch.randn(sd[k].shape, generator=g)
    return HipMlpActorCritic(device=dev, state_dict=sd)


@pytest.mark.gpu
def test_rows_do_not_share_precision():
    """dz1 of every row against float64, with row gradients of one batch spread
    over nine orders of magnitude in random order (40,001 rows: four and five
    tiles per workgroup): a row beside or behind a larger one keeps float32's
    bits.  Bound: sums of up to 192 float32 products through three layers and
    two LayerNorm backwards (differences of like terms) are about 2^-22 of the
    row's norm, some four times that (1e-6) for the worst of 40,001 rows, and as
    much again for another order of the sums: 4e-6."""
    from qqtsim import PPOConfig

    dev, cfg, b = torch.device("cuda:0"), PPOConfig(value_coef=0.0), 40_001
    net = _spread_net(21, dev)

    def scale_rows(adv, ret, old_val):   # (policy term alone: a value error is v's own rounding)
        size = 10.0 ** (-9.0 * torch.rand(adv.shape, generator=torch.Generator().manual_seed(2)))
        adv *= size.to(dev)

    args, z1, w = _smooth_rows(net, b, 21, dev, cfg, 0.0, scale_rows)
    got = {}
    inner = net._l1_weight_grad
    net._l1_weight_grad = lambda x, dz1, *a, **k: got.update(dz1=dz1.clone()) or inner(x, dz1, *a, **k)
    net.ppo_grads(*args, cfg, 0.0)
    x = z1.double().requires_grad_(True)
    (_row_losses(w, x, *args[1:], cfg, 0.0)[0].sum() / b).backward()
    # (rows that the clip or a single legal action leaves without a gradient drop out)
    rows = x.grad.norm(dim=1) > 1e-3 * args[5].abs().double() / b
    assert int(rows.sum()) > b // 4
    err = (got["dz1"].double() - x.grad).norm(dim=1)[rows] / x.grad.norm(dim=1)[rows]
    print(f"worst row {float(err.max()):.2e}, median {float(err.median()):.2e}")
    assert float(err.max()) <= 4e-6


@pytest.mark.gpu
@pytest.mark.parametrize("b", [8193, 40_001])
def test_gradients_of_several_tiles_against_float64(b):
    """Two to five tiles per workgroup, with policy and value outliers of 30
    and 100 times the others in second and later tiles (the earlier tiles still
    matter in every sum), rows within rounding of a kink left out.  Bound: 8
    times the 1.2e-7 that float32 sums of these products show."""
    from qqtsim import PPOConfig

    dev, cfg = torch.device("cuda:0"), PPOConfig()
    net = _spread_net(b, dev)

    def scale_rows(adv, ret, old_val):
        late = torch.arange(8192, adv.numel(), 37, device=dev)
        adv[late[::2]] *= 30.0
        ret[late[1::2]] *= 100.0

    args, z1, w = _smooth_rows(net, b, b, dev, cfg, 0.05, scale_rows)
    net.ppo_grads(*args, cfg, 0.05)
    for v in w.values():
        v.requires_grad_(True)
    x = z1.double() + (w["shared.0.bias"] - w["shared.0.bias"].detach())
    loss, _ = _row_losses(w, x, *args[1:], cfg, 0.05)
    (loss.sum() / b).backward()
    for k, p in net.named_parameters():
        if k != "shared.0.weight":
            err = float((p.grad.double() - w[k].grad).norm() / w[k].grad.norm())
            print(f"{k} {err:.2e}")
            assert err <= 1e-6, (k, err)


@pytest.mark.gpu
def test_parameters_that_view_a_flat_buffer():
    """Parameters at any element of one flat buffer (not 16-byte aligned) are
    served, with the gradients of the same values in tensors of their own."""
    from qqtsim import HipMlpActorCritic, PPOConfig, reference_init

    dev = torch.device("cuda:0")
    sd = reference_init(seed=3)
    args = _case(33, 3, dev, False)
    own, flat = (HipMlpActorCritic(device=dev, state_dict=sd) for _ in range(2))
    buf = torch.zeros(1 + sum(p.numel() + 1 for p in flat.parameters()), device=dev)
    at = 1
    for p in flat.parameters():
        view = buf[at:at + p.numel()].view(p.shape)
        view.copy_(p.detach())
        p.data = view
        at += p.numel() + 1
    assert flat.shared[3].weight.data_ptr() % 16
    for net in (own, flat):
        net.ppo_grads(*args, PPOConfig(), 0.05)
    for (k, p), (_, q) in zip(own.named_parameters(), flat.named_parameters()):
        assert torch.equal(p.grad, q.grad), k


@pytest.mark.gpu
def test_a_refused_call_leaves_the_gradients_alone():
    from qqtsim import HipMlpActorCritic, PPOConfig, reference_init

    dev = torch.device("cuda:0")
    net = HipMlpActorCritic(device=dev, state_dict=reference_init(seed=4))
    args = list(_case(40, 4, dev, False))
    rows = torch.arange(33, device=dev)
    for fill in (None, 3.0):
        for p in net.parameters():
            p.grad = None if fill is None else torch.full_like(p, fill)
        had = [p.grad for p in net.parameters()]
        with pytest.raises(ValueError, match="whole buffer"):
            net.ppo_grads(*args[:-1], args[-1][:33], PPOConfig(), 0.05, rows=rows)
        with pytest.raises(ValueError, match="clip"):
            net.ppo_grads(*args, PPOConfig(clip_eps=-1.0), 0.05, rows=rows)
        assert all(p.grad is g for p, g in zip(net.parameters(), had))
        assert fill is None or all(bool((g == fill).all()) for g in had)


def test_bad_arguments_are_refused():
    from qqtsim import _capi

    lib = _capi.lib()
    a = _capi.PpoStepArgsC()
    assert lib.qqt_ppo_step(ctypes.byref(a), None) == -1
    assert lib.qqt_last_error() == b"qqt_ppo_step: null argument"
    assert lib.qqt_ppo_step_workspace_bytes(0) == -1
    one, many = (lib.qqt_ppo_step_workspace_bytes(n) for n in (1, 1 << 30))
    assert 0 < one < many < 64 << 20
    for name, kind in _capi.PpoStepArgsC._fields_:
        if kind is ctypes.c_void_p:
            setattr(a, name, 4096)
        elif kind is ctypes.c_void_p * 3:
            for i in range(3):
                getattr(a, name)[i] = 4096
    a.batch, a.src_rows, a.workspace_bytes = 1, 1, one
    for field, value, msg in (("batch", 0, b"bad batch"), ("clip_eps", -1.0, b"bad batch"),
                              ("z1", 4100, b"alignment"), ("workspace_bytes", one - 1, b"too small"),
                              ("src_rows", 0, b"row_index")):
        old = getattr(a, field)
        setattr(a, field, value)
        assert lib.qqt_ppo_step(ctypes.byref(a), None) == -1 and msg in lib.qqt_last_error(), field
        setattr(a, field, old)
