"""qqt_ppo_grad (the PPO minibatch with row outputs) through the C ABI against
float64 torch: every row output, the per-block sums, the chunk-transposed
layout and rows read by index (needs an MI355X)."""

from __future__ import annotations

import pytest
import torch

from test_hip_ppo_step import _row_losses, _smooth_rows, _spread_net

pytestmark = pytest.mark.gpu


def _kfrag(m):
    """k-major [K][N] -> the MFMA fragments of qqt_ppo_args: value i of lane
    16 q + r in 16-k group g of column tile t is M[16 g + 4 q + i][16 t + r]."""
    k, n = m.shape
    return m.reshape(k // 16, 4, 4, n // 16, 16).permute(3, 0, 1, 4, 2).contiguous()


def _launch(net, z1, args, cfg, rows=None, t_chunk=0):
    from qqtsim import _capi

    _, mm, bm, act, old_logp, adv, ret, old_val = args
    dev, b = z1.device, z1.shape[0]
    heads = (net.move_head, net.bomb_head, net.critic)
    ln1, l1, ln2 = (net.shared[i] for i in (1, 3, 4))
    cat = lambda i, k: torch.cat([getattr(h[i], k).detach() for h in heads]).contiguous()  # noqa: E731
    w1, wh = l1.weight.detach(), cat(0, "weight")
    ins = dict(z1=z1, ln1_w=ln1.weight, ln1_b=ln1.bias, w1=_kfrag(w1), w1t=_kfrag(w1.t()), b1=l1.bias,
               ln2_w=ln2.weight, ln2_b=ln2.bias, wh=_kfrag(wh), wht=_kfrag(wh.t()), bh=cat(0, "bias"),
               wf=cat(2, "weight"), bf=cat(2, "bias"), actions=act, move_mask=mm.to(torch.uint8),
               bomb_mask=bm.to(torch.uint8), old_logp=old_logp, adv=adv, ret=ret, old_val=old_val)
    n, nb = (-(-b // t_chunk) * t_chunk if t_chunk else b), -(-b // 16)
    shapes = dict(dz1=(b, 128), h1=(n, 128), dz2=(n, 128), h2=(n, 128), hy=(n, 192), dhy=(n, 192),
                  dl=(n, 8), ln_part=(nb, 4, 128), stats_part=(nb, 5), bias_part=(nb, 456),
                  dz1_absmax_part=(nb, 128))
    outs = {k: torch.full(s, float("nan"), device=dev) for k, s in shapes.items()}
    a = _capi.PpoArgsC()
    for k, t in {**ins, **outs}.items():
        assert t.is_contiguous()
        setattr(a, k, t.data_ptr())
    a.batch, a.clip_eps, a.ratio_lo, a.ratio_hi = b, cfg.clip_eps, 1 - cfg.clip_eps, 1 + cfg.clip_eps
    a.value_coef, a.entropy_coef, a.t_chunk = cfg.value_coef, 0.05, t_chunk
    if rows is not None:
        a.row_index, a.src_rows = rows.data_ptr(), act.shape[0]
    _capi.check(_capi.lib().qqt_ppo_grad(a, _capi.stream_handle(dev)))
    torch.cuda.synchronize()
    return outs


@pytest.mark.parametrize("b", [1, 16, 37, 3001])
def test_row_outputs_against_float64(b):
    """Bound: float32 sums of up to 192 products through four layers."""
    from qqtsim import PPOConfig

    dev, cfg = torch.device("cuda:0"), PPOConfig()
    net = _spread_net(b, dev)
    args, z1, w = _smooth_rows(net, b, b, dev, cfg, 0.05, lambda *_: None)
    got = _launch(net, z1, args, cfg)
    ln = torch.nn.functional.layer_norm
    for v in w.values():
        v.requires_grad_(True)
    x = z1.double().requires_grad_(True)
    (_row_losses(w, x, *args[1:], cfg, 0.05)[0].sum() / b).backward()
    h1 = torch.relu(ln(x, (128,), w["shared.1.weight"], w["shared.1.bias"]))
    h2 = torch.relu(ln(h1 @ w["shared.3.weight"].t() + w["shared.3.bias"], (128,),
                       w["shared.4.weight"], w["shared.4.bias"]))
    hy = torch.cat([torch.relu(h2 @ w[f"{h}.0.weight"].t() + w[f"{h}.0.bias"])
                    for h in ("move_head", "bomb_head", "critic")], 1)

    def close(name, a, want):
        err = float((a.double() - want).norm() / want.norm().clamp_min(1e-30))
        assert err <= 3e-6, (name, err)

    close("dz1", got["dz1"], x.grad)
    for k, v in (("h1", h1), ("h2", h2), ("hy", hy)):
        close(k, got[k], v.detach())
    # the weight gradients that the row outputs give a caller
    close("dW1", got["dz2"].double().t() @ got["h1"].double(), w["shared.3.weight"].grad)
    dwh = got["dhy"].double().t() @ got["h2"].double()
    o, bias = 0, got["bias_part"].double().sum(0)
    close("db1", bias[128:256], w["shared.3.bias"].grad)
    close("db0", bias[:128], x.grad.sum(0))
    for i, h in enumerate(("move_head", "bomb_head", "critic")):
        n_out, s = w[f"{h}.2.bias"].numel(), slice(64 * i, 64 * i + 64)
        close(h + " hidden", dwh[s], w[f"{h}.0.weight"].grad)
        close(h + " hidden bias", bias[256:448][s], w[f"{h}.0.bias"].grad)
        close(h + " out", got["dl"][:, o:o + n_out].double().t() @ got["hy"][:, s].double(),
              w[f"{h}.2.weight"].grad)
        close(h + " out bias", bias[448 + o:448 + o + n_out], w[f"{h}.2.bias"].grad)
        o += n_out
    part = got["ln_part"].double().sum(0)
    for i, k in enumerate(("shared.1.weight", "shared.1.bias", "shared.4.weight", "shared.4.bias")):
        close(k, part[i], w[k].grad)
    assert torch.equal(got["dz1_absmax_part"].amax(0), got["dz1"].abs().amax(0))
    assert bool(torch.isfinite(got["stats_part"]).all())


def test_chunk_transposed_and_indexed_rows_equal_the_plain_ones():
    from qqtsim import PPOConfig

    dev, cfg, b, chunk = torch.device("cuda:0"), PPOConfig(), 100, 48
    net = _spread_net(9, dev)
    args, z1, _ = _smooth_rows(net, b, 9, dev, cfg, 0.05, lambda *_: None)
    plain = _launch(net, z1, args, cfg)
    moved = _launch(net, z1, args, cfg, t_chunk=chunk)
    for k in ("dz2", "dhy", "dl"):
        n = plain[k].shape[1]
        rows = moved[k].reshape(-1, n, chunk).transpose(1, 2).reshape(-1, n)
        assert torch.equal(rows[:b], plain[k]), k
    for k in ("dz1", "ln_part", "stats_part", "bias_part", "dz1_absmax_part"):
        assert torch.equal(moved[k], plain[k]), k
    # the per-row inputs in another order, found by index
    perm = torch.randperm(b, device=dev)
    back = torch.argsort(perm)
    shuffled = (None,) + tuple(x[perm].contiguous() for x in args[1:])
    byrow = _launch(net, z1, shuffled, cfg, rows=back)
    for k in plain:
        assert torch.equal(byrow[k], plain[k]), k
