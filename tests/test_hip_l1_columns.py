"""qqt_w0_pack and qqt_l1_grad_columns (the first layer's weight and gradient
with the observation's columns in a player's order) against the same steps in
torch, bit for bit."""

import ctypes

import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("k0", [1, 14, 63, 64, 65, 686, 2366])
def test_weight_fragments(k0):
    from qqtsim.learn import _w0_fragments
    from qqtsim.policy import KBLOCK, _frag

    g = torch.Generator().manual_seed(k0)
    w = torch.randn((128, k0), generator=g).cuda()
    w[3, k0 // 2], w[5, 0], w[127, k0 - 1] = 1e6, 1e-7, float("nan")
    cols = torch.randperm(k0, generator=g).cuda()
    want = _frag(w[:, cols], -(-k0 // KBLOCK) * KBLOCK)
    for x in (w, w.t().contiguous().t(), w.double()):
        got = _w0_fragments(x, cols)
        assert torch.equal(got.isnan(), want.isnan())
        assert torch.equal(got.nan_to_num(0.0), want.nan_to_num(0.0))


@pytest.mark.gpu
@pytest.mark.parametrize("b,k0", [(1, 2), (33, 686), (3600, 2366), (4609, 2366), (40001, 2366)])
def test_gradient_columns(b, k0):
    """Chunk counts below, at and past the reduction's groups of eight.  The
    float64 bound is that of float16 hi/lo pairs without a scale: a low part
    below float16's normal range (2^-14) may be lost."""
    from qqtsim import _capi

    lib, dev = _capi.lib(), torch.device("cuda:0")
    g = torch.Generator().manual_seed(b)
    x = (torch.rand((b, k0), generator=g) < 0.2).half().to(dev)
    dz = torch.randn((b, 128), generator=g).to(dev)
    cols = torch.randperm(k0, generator=g).to(dev)
    need = int(lib.qqt_l1_grad_preferred_floats(b, k0))
    ws = torch.empty(need, device=dev)
    plain, moved = (torch.full((128, k0), float("nan"), device=dev) for _ in range(2))
    a = _capi.L1GradArgsC()
    a.batch, a.k0, a.obs_stride, a.workspace_floats = b, k0, k0, need
    a.obs, a.dz1, a.workspace = x.data_ptr(), dz.data_ptr(), ws.data_ptr()
    a.dw0 = plain.data_ptr()
    _capi.check(lib.qqt_l1_grad(a, _capi.stream_handle(dev)))
    a.dw0 = moved.data_ptr()
    _capi.check(lib.qqt_l1_grad_columns(a, cols.data_ptr(), _capi.stream_handle(dev)))
    assert torch.equal(moved[:, cols], plain)
    want = dz.double().t() @ x.double()
    assert float((plain - want).abs().max()) <= 1e-3 * float(want.abs().max())


def test_bad_arguments_are_refused():
    from qqtsim import _capi

    lib = _capi.lib()
    for args in ((None, 4096, 64, 1, 4096), (4096, None, 64, 1, 4096), (4096, 4096, 64, 1, None),
                 (4096, 4096, 0, 0, 4096), (4096, 4096, 65, 1, 4096), (4096, 4100, 64, 1, 4096),
                 (4096, 4096, 64, 1, 4104)):
        assert lib.qqt_w0_pack(*args, None) == -1 and b"qqt_w0_pack" in lib.qqt_last_error(), args
    a = _capi.L1GradArgsC()
    assert lib.qqt_l1_grad_columns(ctypes.byref(a), 4096, None) == -1
    a.batch, a.k0, a.obs_stride = 8, 64, 64
    a.obs = a.dz1 = a.dw0 = a.workspace = 4096
    a.workspace_floats = lib.qqt_l1_grad_workspace_floats(8, 64)
    for cols in (None, 4100):
        assert lib.qqt_l1_grad_columns(ctypes.byref(a), cols, None) == -1
        assert b"cols must be" in lib.qqt_last_error()


@pytest.mark.gpu
@pytest.mark.parametrize("b,k0", [(1, 126), (31, 128), (33, 130), (513, 2432), (8192, 2560),
                                  (9000, 258), (70_001, 1024), (70_001, 1026)])
def test_narrow_and_wide_column_tiles(b, k0):
    """Edges of the 128- and 512-column tiles and both sides of the rule that
    picks them (1024 columns in 64 chunks: 128 wide tiles; 1026: 192), against
    float64.  float16 pairs of a gradient scaled to 2^14 hold 22 bits."""
    from qqtsim import _capi

    lib, dev = _capi.lib(), torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(b + k0)
    x = (torch.rand((b, k0 + 2), generator=g, device=dev) < 0.2).half()[:, :k0]
    dz = torch.randn((b, 128), generator=g, device=dev)
    scale = torch.exp2(13.0 - torch.ceil(torch.log2(dz.abs().max()))).reshape(1)
    cols = torch.arange(k0, device=dev)
    need = int(lib.qqt_l1_grad_preferred_floats(b, k0))
    ws, out = torch.empty(need, device=dev), torch.full((128, k0), float("nan"), device=dev)
    a = _capi.L1GradArgsC()
    a.batch, a.k0, a.obs_stride, a.workspace_floats = b, k0, k0 + 2, need
    a.obs, a.dz1, a.dz_scale = x.data_ptr(), dz.data_ptr(), scale.data_ptr()
    a.workspace, a.dw0 = ws.data_ptr(), out.data_ptr()
    _capi.check(lib.qqt_l1_grad_columns(a, cols.data_ptr(), _capi.stream_handle(dev)))
    want = dz.double().t() @ x.double()
    assert float((out - want).norm()) <= 2e-6 * float(want.norm())


@pytest.mark.gpu
@pytest.mark.parametrize("b,k0", [(1, 130), (33, 2366), (30_001, 2366)])
def test_a_non_finite_last_row_stays_its_own(b, k0):
    """An infinity and a NaN in the batch's last row reach dW0 as that row's
    products alone: infinite with the gradient's sign, NaN where the entry is
    NaN, the other columns finite (both column tiles; the last step of the
    batch is partial).  That row's gradients have a high and a low part of one
    sign, whose two products of an infinity do not cancel."""
    from qqtsim import _capi

    lib, dev = _capi.lib(), torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(b)
    x = (torch.rand((b, k0), generator=g, device=dev) < 0.2).half()
    x[-1, 1], x[-1, 3], x[-1, k0 - 1] = float("inf"), float("nan"), float("-inf")
    dz = torch.randn((b, 128), generator=g, device=dev)
    dz[-1] = (1.0 + 2.0 ** -12) * dz[-1].sign()
    need = int(lib.qqt_l1_grad_preferred_floats(b, k0))
    ws, out = torch.empty(need, device=dev), torch.empty((128, k0), device=dev)
    a = _capi.L1GradArgsC()
    a.batch, a.k0, a.obs_stride, a.workspace_floats = b, k0, k0, need
    a.obs, a.dz1, a.workspace, a.dw0 = (t.data_ptr() for t in (x, dz, ws, out))
    _capi.check(lib.qqt_l1_grad(a, _capi.stream_handle(dev)))
    assert torch.equal(out[:, 1], float("inf") * dz[-1].sign())
    assert torch.equal(out[:, k0 - 1], -float("inf") * dz[-1].sign())
    assert bool(out[:, 3].isnan().all())
    assert torch.isfinite(out).all(0).sum() == k0 - 3
