"""Partial column sums that the wide backward kernels leave: every column once, at the edges of the row variants."""
import ctypes

import pytest
import torch

from test_gpu_parity import DEV, assert_grad_close, rand_bf16

pytestmark = pytest.mark.gpu


# first and last width of the row variants, full ones, rows that end inside a 16-byte group of a wave's share of the sums
@pytest.mark.parametrize("cols", [264, 512, 520, 1000, 1024, 1032, 1536, 1544, 2048, 2056, 3072, 3080, 4096, 4104, 5120,
                                  5128, 6144, 6152, 8192, 8200, 12288, 12296, 16384, 16392, 32760, 32768])
@pytest.mark.parametrize("rows", [1, 37, 700])
def test_partials_cover_each_column_once(lib, cols, rows):
    x, dy = (rand_bf16(rows, cols, seed=i).to(DEV) for i in range(2))
    p = rand_bf16(cols, seed=2, scale=0.2).to(DEV)
    dx = torch.empty_like(x)
    st = torch.cuda.current_stream().cuda_stream
    xd, d = x.double(), dy.double()
    dev = xd - xd.mean(-1, keepdim=True)
    xh = dev * torch.rsqrt(dev.square().mean(-1, keepdim=True) + 1e-6)
    xr = xd * torch.rsqrt(xd.square().mean(-1, keepdim=True) + 1e-6)
    for n_acc, need, refs in ((2, lib.tt_adaln_backward_workspace_bytes(rows, cols, rows), (d * xh, d)),
                              (1, lib.tt_rmsnorm_backward_workspace_bytes(rows, cols), (d * xr,))):
        ws = torch.full((need // 4 + 64,), 1e30, device=DEV)
        n = ctypes.c_int(0)
        args = (dx.data_ptr(), dy.data_ptr(), x.data_ptr(), p.data_ptr(), ws.data_ptr(), need, ctypes.byref(n), rows, cols)
        assert (lib.tt_adaln_backward_partials(*args, rows, 1e-6, st) if n_acc == 2 else
                lib.tt_rmsnorm_backward_partials(*args, 1e-6, st)) == 0
        torch.cuda.synchronize()
        used = n.value * n_acc * cols
        assert (ws[used:] == 1e30).all()
        sums = ws[:used].view(n.value, n_acc, cols).double().sum(0)
        for got, ref, name in zip(sums, refs, ("first", "second")):
            assert_grad_close(got, ref.sum(0).cpu(), rows, f"{name} sums, {n.value} partials")


@pytest.mark.parametrize("cols", [520, 1536, 3080, 5120, 8200, 16392])
def test_gate_and_residual_gradients(cols):
    from teletron_amd import ops
    rows, eps = 411, 1e-6
    x, r, dy, ds = (rand_bf16(rows, cols, seed=i).to(DEV) for i in range(4))
    gate, scale = (rand_bf16(1, cols, seed=4 + i, scale=0.2).to(DEV) for i in range(2))
    _, dg = ops.gate_residual_backward(dy, gate, r)
    assert_grad_close(dg, (dy.double() * r.double()).sum(0).cpu(), rows, "dgate")
    _, _, dscale, dshift, dgate = ops.residual_norm_backward(dy, ds, x, r, gate, scale, eps, False)
    xd, d = x.double(), dy.double()
    dev = xd - xd.mean(-1, keepdim=True)
    rstd = torch.rsqrt(dev.square().mean(-1, keepdim=True) + eps)
    xh, g = dev * rstd, d * (1 + scale.double())
    dx = ds.double() + rstd * (g - g.mean(-1, keepdim=True) - xh * (g * xh).mean(-1, keepdim=True))
    for got, ref, name in ((dscale, d * xh, "dscale"), (dshift, d, "dshift"), (dgate, dx * r.double(), "dgate of the update")):
        assert_grad_close(got, ref.sum(0).cpu(), rows, name)


# rounds of 8 x 16 and 8 x 32 partials, a last one of a single partial, column counts beside whole workgroups of 32 and 64
@pytest.mark.parametrize("n_partials", [1, 31, 33, 128, 129, 256, 257, 777])
@pytest.mark.parametrize("n_batches,cols", [(1, 1), (1, 33), (1, 128), (1, 4600), (1, 4616), (1, 5128), (2, 8191), (3, 5120), (300, 72), (70, 300)])
@pytest.mark.parametrize("n_acc", [1, 2])
def test_reduction(lib, n_partials, n_batches, cols, n_acc):
    """Any order of n additions is off by at most n 2^-24 sum |x|."""
    g = torch.Generator(device=DEV).manual_seed(n_partials + cols)
    ws = torch.randn(n_batches, n_partials, n_acc, cols, generator=g, device=DEV)
    out = torch.full((n_acc, n_batches, cols), float("nan"), device=DEV)
    assert lib.tt_reduce_partials(out[0].data_ptr(), out[1].data_ptr() if n_acc == 2 else None, ws.data_ptr(), n_batches,
                                  n_partials, n_acc, cols, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    d = ws.double()
    err = (out.double().transpose(0, 1) - d.sum(1)).abs()
    assert (err <= n_partials * 2.0 ** -24 * d.abs().sum(1)).all()
