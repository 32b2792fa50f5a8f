"""qqt_lstm_seq_forward / _backward (the lstm learner's recurrence over whole
sequences) against the frame-by-frame recurrence in float64 torch."""

from __future__ import annotations

import ctypes

import pytest
import torch

HID = 128


def _frame_by_frame(x, lstm, keep, window):
    """The update's recurrence (train/ppo.py:463-490) from the module's
    weights in float64: outputs (T, m, 128)."""
    h = c = torch.zeros((x.shape[1], HID), dtype=x.dtype, device=x.device)
    outs = []
    for t in range(x.shape[0]):
        if window > 0 and t % window == 0:
            h, c = h.detach(), c.detach()
        z = (x[t] @ lstm.weight_ih_l0.t() + lstm.bias_ih_l0 + h @ lstm.weight_hh_l0.t()
             + lstm.bias_hh_l0)
        i, f, g, o = z.chunk(4, -1)
        c = torch.sigmoid(f) * c + torch.sigmoid(i) * torch.tanh(g)
        h = torch.sigmoid(o) * torch.tanh(c)
        outs.append(h)
        h, c = h * keep[t][:, None], c * keep[t][:, None]
    return torch.stack(outs)


@pytest.mark.gpu
@pytest.mark.parametrize("steps,m,window", [(1, 1, 0), (2, 15, 0), (7, 16, 3), (33, 17, 8),
                                            (8, 31, 1), (32, 256, 0), (128, 37, 16)])
def test_sequence_kernels_match_the_frame_by_frame_recurrence(steps, m, window):
    from qqtsim.learn import _sequence_kernels_serve, _sequence_outputs

    torch.manual_seed(steps * 1000 + m)
    lstm = torch.nn.LSTM(256, HID, batch_first=True).cuda()
    x = torch.randn(steps, m, 256, device="cuda").relu().requires_grad_(True)
    keep = (torch.rand(steps, m, device="cuda") > 0.1).float()
    dy = torch.randn(steps, m, HID, device="cuda")
    assert _sequence_kernels_serve(lstm, x)
    out = _sequence_outputs(lstm, x, keep, window)
    out.backward(dy)
    ref = torch.nn.LSTM(256, HID, batch_first=True).cuda().double()
    ref.load_state_dict({k: v.double() for k, v in lstm.state_dict().items()})
    x64 = x.detach().double().requires_grad_(True)
    want = _frame_by_frame(x64, ref, keep.double(), window)
    want.backward(dy.double())

    def rel(a, b):
        return float((a.double() - b).norm() / b.norm().clamp_min(1e-30))

    # float32 sums of up to 512 terms and steps m rows: a few times
    # sqrt(512) 2^-24 = 1.3e-6 per product, carried through the frames
    assert rel(out, want) < 2e-6
    assert rel(x.grad, x64.grad) < 5e-6
    for (k, p), (_, q) in zip(lstm.named_parameters(), ref.named_parameters()):
        assert rel(p.grad, q.grad) < 5e-6, k


@pytest.mark.gpu
@pytest.mark.parametrize("steps,m", [(12, 37), (32, 256), (24, 1400)])
def test_weight_gradients_keep_the_precision_of_frame_products(steps, m):
    """dW_ih, dW_hh and the input gradient are no further from float64 than
    nn.LSTM called frame by frame is (the update's path for modules that the
    sequence kernels do not serve).  Bound: 1.25 times its error, for sums in
    another order; one sum over 4,096 rows is at four times."""
    from qqtsim.learn import _sequence_outputs

    torch.manual_seed(steps + m)
    lstm = torch.nn.LSTM(256, HID, batch_first=True).cuda()
    base = torch.randn(steps, m, 256, device="cuda").relu()
    keep = (torch.rand(steps, m, device="cuda") > 0.05).float()
    dy = torch.randn(steps, m, HID, device="cuda")

    def by_module(x, net):
        state, outs = None, []
        for t in range(steps):
            out, state = net(x[t].unsqueeze(1), state)
            outs.append(out.squeeze(1))
            state = tuple(v * keep[t][:, None].to(v.dtype) for v in state)
        return torch.stack(outs)

    def grads(run, dtype):
        net = torch.nn.LSTM(256, HID, batch_first=True).cuda().to(dtype)
        net.load_state_dict({k: v.to(dtype) for k, v in lstm.state_dict().items()})
        x = base.to(dtype).clone().requires_grad_(True)
        run(x, net).backward(dy.to(dtype))
        return dict(ih=net.weight_ih_l0.grad, hh=net.weight_hh_l0.grad, x=x.grad)

    want = grads(lambda x, net: _frame_by_frame(x, net, keep.double(), 0), torch.float64)
    got = grads(lambda x, net: _sequence_outputs(net, x, keep, 0), torch.float32)
    module = grads(by_module, torch.float32)
    for k, w in want.items():
        mine, theirs = (float((g[k].double() - w).norm() / w.norm()) for g in (got, module))
        print(f"{k}: {mine:.2e}, frame by frame {theirs:.2e}")
        assert mine <= 1.25 * theirs, k


@pytest.mark.gpu
def test_weights_and_saved_tensors_at_any_element():
    """W_hh as a view into a flat buffer, and tensors that a saved-tensor hook
    hands back at an odd element: the gradients of the plain call."""
    from qqtsim.learn import _sequence_outputs

    torch.manual_seed(5)
    steps, m = 5, 19
    x = torch.randn(steps, m, 256, device="cuda")
    keep = (torch.rand(steps, m, device="cuda") > 0.2).float()
    dy = torch.randn(steps, m, HID, device="cuda")
    plain = torch.nn.LSTM(256, HID, batch_first=True).cuda()
    moved = torch.nn.LSTM(256, HID, batch_first=True).cuda()
    for k in ("weight_ih_l0", "weight_hh_l0", "bias_ih_l0", "bias_hh_l0"):
        p = getattr(plain, k).detach()
        view = torch.zeros(p.numel() + 1, device="cuda")[1:].view(p.shape)
        getattr(moved, k).data = view.copy_(p)
    assert moved.weight_hh_l0.data_ptr() % 16

    def pack(t):
        return torch.cat([t.new_zeros(1), t.detach().reshape(-1)]), t.shape

    _sequence_outputs(plain, x, keep, 2).backward(dy)
    with torch.autograd.graph.saved_tensors_hooks(pack, lambda s: s[0][1:].view(s[1])):
        _sequence_outputs(moved, x, keep, 2).backward(dy)
    for (k, p), (_, q) in zip(plain.named_parameters(), moved.named_parameters()):
        assert torch.equal(p.grad, q.grad), k


def test_only_a_plain_float32_lstm_on_the_gpu_is_served():
    from qqtsim.learn import _sequence_kernels_serve

    class Lstm(torch.nn.LSTM):
        pass

    x = torch.zeros(2, 3, 256)
    assert not _sequence_kernels_serve(torch.nn.LSTM(256, HID, batch_first=True), x)
    assert not _sequence_kernels_serve(Lstm(256, HID, batch_first=True), x)
    if torch.cuda.is_available():
        x = x.cuda()
        lstm = torch.nn.LSTM(256, HID, batch_first=True).cuda()
        assert _sequence_kernels_serve(lstm, x)
        hook = lstm.register_forward_hook(lambda *a: None)
        assert not _sequence_kernels_serve(lstm, x)
        hook.remove()
        assert not _sequence_kernels_serve(lstm.double(), x)


def test_bad_arguments_are_refused():
    from qqtsim import _capi

    lib = _capi.lib()
    for fn, own in ((lib.qqt_lstm_seq_forward, ("zx", "h")), (lib.qqt_lstm_seq_backward, ("dh", "dz"))):
        def args():
            a = _capi.LstmSeqArgsC(steps=4, rows=3)
            for k in ("w_hh", "keep", "c", "gates") + own:
                setattr(a, k, 4096)
            return a
        for k in ("w_hh", "keep", "c", "gates") + own:
            a = args()
            setattr(a, k, None)
            assert fn(ctypes.byref(a), None) == -1 and b"null argument" in lib.qqt_last_error(), k
        for k, v in (("steps", 0), ("rows", -1), ("window", -1), ("w_hh", 4100)):
            a = args()
            setattr(a, k, v)
            assert fn(ctypes.byref(a), None) == -1 and b"bad steps" in lib.qqt_last_error(), k
