"""Rows of any length and tensors at any 2-byte address: which kernels a call runs on, and that this and
every bit of the result depend on its arguments alone.  Tolerances as in test_gpu_parity.py."""
import pytest
import torch

from test_gpu_parity import DEV, rand_bf16

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
