"""Wide rows that are not whole 128-byte lines (cols % 64 != 0): the lines that neighbouring waves and
rows share are stored another way than the rest, so every segment edge of every variant is checked,
and that nothing is written beside the rows.  Tolerances as in test_gpu_parity.py."""
import pytest
import torch

from test_gpu_gate import test_gate_residual_shapes as check_gate
from test_gpu_parity import DEV, check_adaln, check_rmsnorm, rand_bf16
from test_gpu_resnorm import run_case as check_residual

pytestmark = pytest.mark.gpu

# the shortest and the longest ragged row of each variant (lane slots 64 ... 4096 packs of 8)
SLOTS = [32, 64, 128, 192, 256, 384, 512, 640, 768, 1024, 1536, 2048, 4096]
WIDTHS = [8 * w for lo, hi in zip(SLOTS, SLOTS[1:]) for w in (lo + 1, hi - 1)]


@pytest.mark.parametrize("cols", WIDTHS)
def test_ragged_widths(cols):
    nb, rpb = 2, 19
    x, dy = rand_bf16(nb, rpb, cols, seed=cols), rand_bf16(nb, rpb, cols, seed=cols + 1)
    p = [rand_bf16(nb, 1, cols, seed=cols + 2 + i, scale=0.2) for i in range(2)]
    check_adaln(x, p[0], p[1], dy, 1e-6, nb, f"cols {cols}")
    check_rmsnorm(x, 1 + p[0][0, 0], dy, 1e-6, f"cols {cols}")
    check_gate(cols, nb, rpb)
    for gated in (False, True):
        check_residual(cols, nb, rpb, gated, affine=False)


@pytest.mark.parametrize("cols", [1000, 3688])
@pytest.mark.parametrize("shift", range(0, 64, 8))
def test_ragged_rows_at_any_16_byte_offset(lib, cols, shift):
    """The same bits wherever in a line the tensors start, and the values around them untouched."""
    rows, guard, eps = 23, 256, 1e-6
    x, dy = (rand_bf16(rows, cols, seed=cols + i).to(DEV) for i in range(2))
    w, b = (rand_bf16(cols, seed=cols + 2 + i, scale=0.2).to(DEV) for i in range(2))

    def placed(t, s):
        buf = torch.full((t.numel() + 2 * guard,), 7.0, dtype=t.dtype, device=DEV)
        buf[guard + s:guard + s + t.numel()] = t.flatten()
        return buf, buf.data_ptr() + 2 * (guard + s)

    def run(s):
        bufs = {}
        for name, t in (("x", x), ("dy", dy), ("y", torch.zeros_like(x)), ("dx", torch.zeros_like(x)),
                        ("s", torch.zeros_like(x)), ("g", torch.zeros_like(x))):
            bufs[name] = placed(t, s)
        ptr = {k: v[1] for k, v in bufs.items()}
        grads = torch.zeros(2, cols, device=DEV)
        ws = torch.empty(lib.tt_adaln_backward_workspace_bytes(rows, cols, rows), dtype=torch.uint8, device=DEV)
        stream = torch.cuda.current_stream().cuda_stream
        assert lib.tt_adaln_backward(ptr["dx"], grads[0].data_ptr(), grads[1].data_ptr(), ptr["dy"], ptr["x"], w.data_ptr(),
                                     ws.data_ptr(), ws.numel(), rows, cols, rows, eps, stream) == 0
        assert lib.tt_residual_norm_forward(ptr["s"], ptr["y"], ptr["x"], ptr["dy"], None, 1, w.data_ptr(), b.data_ptr(), 1, 0,
                                            None, None, rows, cols, rows, eps, stream) == 0
        assert lib.tt_gate_residual_forward(ptr["g"], ptr["x"], w.data_ptr(), ptr["dy"], rows, cols, rows, stream) == 0
        torch.cuda.synchronize()
        out = [grads]
        for name in ("y", "dx", "s", "g"):
            buf = bufs[name][0]
            assert (buf[:guard + s] == 7).all() and (buf[guard + s + x.numel():] == 7).all(), name
            out.append(buf[guard + s:guard + s + x.numel()])
        return out

    for got, want in zip(run(shift), run(0)):
        assert torch.equal(got, want)


# one value more than a variant of the kernels holds, one less, and a short last pack of every length
ODD = [257, 511, 513, 1001, 1023, 1535, 1537, 2049, 3073, 4095, 5121, 6143, 8193, 16383, 32767] + list(range(521, 528))


@pytest.mark.parametrize("cols", ODD)
def test_odd_widths(cols):
    for nb, rpb in ((1, 1), (2, 37), (41, 1)):
        x, dy = rand_bf16(nb, rpb, cols, seed=cols), rand_bf16(nb, rpb, cols, seed=cols + 1)
        p = [rand_bf16(nb, 1, cols, seed=cols + 2 + i, scale=0.2) for i in range(2)]
        check_adaln(3 + x, p[0], p[1], dy, 1e-6, nb, f"cols {cols}")
        check_rmsnorm(x, 1 + p[0][0, 0], dy, 1e-6, f"cols {cols}")


@pytest.mark.parametrize("cols", [1001, 1000, 1536])
@pytest.mark.parametrize("shift", [1, 3, 8, 13])
def test_backward_at_any_address_and_workspace(lib, cols, shift):
    """Nothing beside the rows and gradients is written; the smallest workspace (two floats a row, with
    which the element-wise kernels run) gives the same gradients."""
    rows, guard = 2500, 64
    x, dy, w = rand_bf16(rows, cols, seed=1), rand_bf16(rows, cols, seed=2), rand_bf16(cols, seed=3, scale=0.2)
    from oracle import norm_oracle as O
    from test_gpu_parity import assert_bf16_close, assert_grad_close
    dxo, dso, dho = O.adaln_backward(dy, x, w, 1e-6, 1)

    def placed(t):
        buf = torch.full((t.numel() + 2 * guard,), 7.0, dtype=t.dtype, device=DEV)
        buf[guard + shift:guard + shift + t.numel()] = t.flatten().to(DEV)
        return buf, buf.data_ptr() + 2 * (guard + shift)

    (xb, xp), (db, dp), (wb, wp), (ob, op) = (placed(t) for t in (x, dy, w, torch.zeros_like(x)))
    stream = torch.cuda.current_stream().cuda_stream
    need = max(lib.tt_adaln_backward_workspace_bytes(rows, cols, rows), rows * 8)
    for size, status in ((need, 0), (rows * 8, 0), (rows * 8 - 4, 3)):
        if shift == 8 and cols % 8 == 0 and size != need:
            continue                                   # 16-byte aligned: the ordinary kernels, which need it all
        ws = torch.full((size // 4 + guard,), 5.0, device=DEV)
        grads = torch.full((2, cols + guard), 5.0, device=DEV)
        assert lib.tt_adaln_backward(op, grads[0].data_ptr(), grads[1].data_ptr(), dp, xp, wp, ws.data_ptr(), size,
                                     rows, cols, rows, 1e-6, stream) == status
        torch.cuda.synchronize()
        assert (ws[size // 4:] == 5).all() and (grads[:, cols:] == 5).all()
        assert (ob[:guard + shift] == 7).all() and (ob[guard + shift + x.numel():] == 7).all()
        if status == 0:
            assert_bf16_close(ob[guard + shift:guard + shift + x.numel()], dxo, "dx")
            assert_grad_close(grads[0, :cols], dso, rows, "dscale")
            assert_grad_close(grads[1, :cols], dho, rows, "dshift")


@pytest.mark.parametrize("cols,batches", [(5128, 2), (6136, 2), (2200, 1), (1000, 1)])
def test_static_scratch_takes_ragged_tensors(lib, cols, batches):
    """The kernels of ragged rows may keep twice the workgroups of the masked ones resident; where the partial
    sums of all batches are too large for the scratch array (5128 and 6136 columns) they go through it batch by
    batch, with the same bits."""
    from teletron_amd import cabi, ops
    rows = 1000 * batches
    need = lib.tt_adaln_backward_workspace_bytes(rows, cols, 1000)
    assert (need > cabi.TT_STATIC_WORKSPACE_BYTES) == (batches == 2)
    x, dy = (rand_bf16(rows, cols, seed=i).to(DEV) for i in range(2))
    w = rand_bf16(batches, cols, seed=2, scale=0.2).to(DEV)
    dx, ds, dh = ops.adaln_backward(dy, x, w, 1e-6)
    dx2, g = torch.empty_like(dx), torch.empty(2, batches, cols, device=DEV)
    assert lib.tt_adaln_backward_static(dx2.data_ptr(), g[0].data_ptr(), g[1].data_ptr(), dy.data_ptr(), x.data_ptr(),
                                        w.data_ptr(), rows, cols, 1000, 1e-6, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    assert torch.equal(dx, dx2)
    assert torch.equal(g[0], ds) and torch.equal(g[1], dh)
