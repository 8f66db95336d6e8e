"""Rows of any length and tensors at any 2-byte address: which kernels a call runs on, and that this and
every bit of the result depend on its arguments alone.  Tolerances as in test_gpu_parity.py."""
import pytest
import torch

from test_gpu_configs import whole_tensor_check
from test_gpu_parity import DEV, assert_grad_close, rand_bf16

pytestmark = pytest.mark.gpu


def shifted(t, by):
    """The values of ``t`` in a buffer of their own, ``by`` values behind a 16-byte boundary."""
    buf = torch.empty(t.numel() + by, dtype=t.dtype, device=DEV)
    buf[by:] = t.flatten().to(DEV)
    return buf[by:].view(t.shape)


# shapes whose aligned AdaLN kernel takes two rows a tile and so asks for fewer partial sums, and one that does not
@pytest.mark.parametrize("nb,rpb,cols", [(2, 512, 1536), (1, 2500, 1536), (3, 700, 1000), (1, 1500, 3072), (1, 900, 5120)])
def test_misaligned_backward_does_not_depend_on_earlier_calls(lib, nb, rpb, cols):
    from teletron_amd import ops
    rows = nb * rpb
    x, dy = (shifted(rand_bf16(rows, cols, seed=i), 3) for i in range(2))
    w = shifted(rand_bf16(nb, cols, seed=2, scale=0.2), 5)
    calls = [lambda: ops.adaln_backward(dy, x, w, 1e-6), lambda: ops.rmsnorm_backward(dy, x, w[0], 1e-6)]
    ops.clear_workspaces()
    first = [call() for call in calls]
    big = rand_bf16(8000, 8192, seed=3).to(DEV)
    ops.adaln_backward(big, big, big[0], 1e-6)              # leaves a workspace with room to spare
    for call, want in zip(calls, first):
        for a, b in zip(call(), want):
            assert torch.equal(a, b)

    # the workspace that the queries ask for holds the partial sums of the vector kernels: they are
    # written behind the two floats a row that the element-wise kernels keep
    st = torch.cuda.current_stream().cuda_stream
    dx, g = torch.empty_like(x), torch.empty(2, nb, cols, device=DEV)
    for name, need in (("adaln", lib.tt_adaln_backward_workspace_bytes(rows, cols, rpb)),
                       ("rms", lib.tt_rmsnorm_backward_workspace_bytes(rows, cols))):
        assert need > 2 * rows * 8
        ws = torch.full((need // 4,), 1e30, device=DEV)
        if name == "adaln":
            rc = lib.tt_adaln_backward(dx.data_ptr(), g[0].data_ptr(), g[1].data_ptr(), dy.data_ptr(), x.data_ptr(),
                                       w.data_ptr(), ws.data_ptr(), need, rows, cols, rpb, 1e-6, st)
        else:
            rc = lib.tt_rmsnorm_backward(dx.data_ptr(), g[0].data_ptr(), dy.data_ptr(), x.data_ptr(), w.data_ptr(),
                                         ws.data_ptr(), need, rows, cols, 1e-6, st)
        assert rc == 0
        torch.cuda.synchronize()
        assert (ws[rows * 2:] != 1e30).any(), name


@pytest.mark.parametrize("cols", [250, 257, 1001, 16383, 16385, 32767])
def test_odd_widths_run_on_the_faster_kernels(lib, cols):
    """The vector kernels leave partial sums in the workspace, the element-wise ones two floats a row."""
    rows, st = 700, torch.cuda.current_stream().cuda_stream
    x, dy = (rand_bf16(rows, cols, seed=i).to(DEV) for i in range(2))
    w = rand_bf16(cols, seed=2, scale=0.2).to(DEV)
    vector = 256 < cols <= 16384
    dx, g = torch.empty_like(x), torch.empty(2, cols, device=DEV)
    for adaln, need in ((True, lib.tt_adaln_backward_workspace_bytes(rows, cols, rows)),
                        (False, lib.tt_rmsnorm_backward_workspace_bytes(rows, cols))):
        assert (need > rows * 8) == vector
        ws = torch.full((1 << 24,), 1e30, device=DEV)
        args = [dy.data_ptr(), x.data_ptr(), w.data_ptr(), ws.data_ptr(), ws.numel() * 4, rows, cols]
        if adaln:
            assert lib.tt_adaln_backward(dx.data_ptr(), g[0].data_ptr(), g[1].data_ptr(), *args, rows, 1e-6, st) == 0
        else:
            assert lib.tt_rmsnorm_backward(dx.data_ptr(), g[0].data_ptr(), *args, 1e-6, st) == 0
        torch.cuda.synchronize()
        assert (ws[:rows * 2] != 1e30).all() and (ws[rows * 2:need // 4] != 1e30).any() == vector
        assert (ws[need // 4:] == 1e30).all()


# partial sums of all batches, or of one, that exceed the scratch array of tt_adaln_backward_static: ragged and odd
# rows, misaligned ones (shift), and a modulation vector for every few rows
@pytest.mark.parametrize("nb,rpb,cols,shift", [(2, 1000, 5128, 0), (1, 3000, 5128, 0), (1, 3000, 8184, 0), (3, 500, 6136, 0),
                                               (1, 3000, 5127, 0), (2, 700, 8191, 0), (1, 900, 16383, 0), (1, 300, 32767, 0),
                                               (5, 60, 32767, 0), (300, 10, 8191, 0), (3000, 2, 1001, 0),
                                               (1, 3000, 5120, 3), (2, 900, 8192, 1), (1, 500, 16384, 4)])
def test_static_backward_equals_the_workspace_backward(lib, nb, rpb, cols, shift):
    rows = nb * rpb
    x, dy = (shifted(rand_bf16(rows, cols, seed=i), shift) for i in range(2))
    w = rand_bf16(nb, cols, seed=2, scale=0.2).to(DEV)
    need = max(lib.tt_adaln_backward_workspace_bytes(rows, cols, rpb), rows * 8)
    ws = torch.empty(need, dtype=torch.uint8, device=DEV)
    st = torch.cuda.current_stream().cuda_stream
    out = [[torch.full_like(x, float("nan")), torch.full((2, nb, cols), float("nan"), device=DEV)] for _ in range(2)]
    (a, ga), (b, gb) = out
    assert lib.tt_adaln_backward(a.data_ptr(), ga[0].data_ptr(), ga[1].data_ptr(), dy.data_ptr(), x.data_ptr(), w.data_ptr(),
                                 ws.data_ptr(), need, rows, cols, rpb, 1e-6, st) == 0
    for _ in range(2):                          # the array is left as the first call filled it
        assert lib.tt_adaln_backward_static(b.data_ptr(), gb[0].data_ptr(), gb[1].data_ptr(), dy.data_ptr(), x.data_ptr(),
                                            w.data_ptr(), rows, cols, rpb, 1e-6, st) == 0
        torch.cuda.synchronize()
        assert torch.equal(a, b) and torch.equal(ga, gb)


@pytest.mark.parametrize("rows,cols,shift", [(30000, 257, 0), (9000, 1001, 0), (7001, 4095, 0), (1300, 16383, 0), (9000, 1536, 3),
                                             (140000, 257, 0), (36000, 1001, 0), (24000, 1536, 5), (2100, 16383, 0), (1100, 32767, 0)])
def test_many_odd_rows(lib, rows, cols, shift):
    """Several tiles a workgroup, in the caches and (from the sixth case) past the 64 MiB where the plans change:
    every element against torch fp32 on the GPU, the parameter gradients against fp64 sums."""
    from teletron_amd import ops
    nb, eps = 2 if rows % 2 == 0 else 1, 1e-6
    g = torch.Generator(device=DEV).manual_seed(cols)
    x, dy = (shifted(torch.randn(rows, cols, generator=g, device=DEV).to(torch.bfloat16), shift) for _ in range(2))
    p = (0.2 * torch.randn(2, nb, cols, generator=g, device=DEV)).to(torch.bfloat16)
    w = (1 + p[0, 0].float()).to(torch.bfloat16)
    group = torch.arange(rows, device=DEV) // (rows // nb)

    y, mean, rstd = ops.adaln_forward(x, p[0], p[1], eps, return_stats=True)
    yr = ops.rmsnorm_forward(x, w, eps)
    y2, xn, inv = torch.empty_like(x), torch.empty_like(x), torch.empty(rows, device=DEV)
    st = torch.cuda.current_stream().cuda_stream
    assert lib.tt_launch_adaln_forward(y2.data_ptr(), xn.data_ptr(), x.data_ptr(), p[0, 0].data_ptr(), p[1, 0].data_ptr(),
                                       rows, cols, eps, inv.data_ptr(), st) == 0
    dx, ds, dh = ops.adaln_backward(dy, x, p[0], eps)
    dxr, dw = ops.rmsnorm_backward(dy, x, w, eps)

    def parts(r0, r1):
        xs = x[r0:r1].float()
        d = xs - xs.mean(-1, keepdim=True)
        return d * torch.rsqrt(d.pow(2).mean(-1, keepdim=True) + eps), torch.rsqrt(d.pow(2).mean(-1, keepdim=True) + eps), \
            xs * torch.rsqrt(xs.pow(2).mean(-1, keepdim=True) + eps), torch.rsqrt(xs.pow(2).mean(-1, keepdim=True) + eps)

    def grad(r0, r1, k, gg):
        xh, rs = parts(r0, r1)[k:k + 2]
        return rs * (gg - (gg.mean(-1, keepdim=True) if k == 0 else 0) - xh * (gg * xh).mean(-1, keepdim=True))

    scale, shift_ = 1 + p[0].float(), p[1].float()
    whole_tensor_check(y, lambda a, b: parts(a, b)[0] * scale[group[a:b]] + shift_[group[a:b]])
    whole_tensor_check(yr, lambda a, b: parts(a, b)[2] * w.float())
    whole_tensor_check(xn, lambda a, b: parts(a, b)[0])
    whole_tensor_check(y2, lambda a, b: parts(a, b)[0] * scale[0] + shift_[0])
    whole_tensor_check(dx, lambda a, b: grad(a, b, 0, dy[a:b].float() * scale[group[a:b]]))
    whole_tensor_check(dxr, lambda a, b: grad(a, b, 2, dy[a:b].float() * w.float()))
    sums = torch.zeros(3, nb, cols, dtype=torch.float64, device=DEV)
    for a in range(0, rows, 8192):
        b = min(a + 8192, rows)
        xh, rs, xr, _ = parts(a, b)
        d = dy[a:b].double()
        for i, t in enumerate((d * xh.double(), d, d * xr.double())):
            sums[i].index_add_(0, group[a:b], t)
        torch.testing.assert_close(rstd[a:b], rs[:, 0], rtol=1e-5, atol=0)
    assert torch.equal(rstd, inv)
    assert_grad_close(ds, sums[0].cpu(), rows, "dscale")
    assert_grad_close(dh, sums[1].cpu(), rows, "dshift")
    assert_grad_close(dw, sums[2].sum(0).cpu(), rows, "dweight")
