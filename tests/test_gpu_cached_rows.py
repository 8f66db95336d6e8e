"""Tensors that fit the caches are read by kernels of their own: the same bits a row as from the streaming ones."""
import pytest
import torch

from test_gpu_parity import DEV

pytestmark = pytest.mark.gpu
EPS = 1e-6


# full rows, masked ones of whole cache lines, ragged ones (with many, some and few idle lanes, and past the short variants), narrow rows
@pytest.mark.parametrize("cols", [512, 520, 776, 1000, 1288, 1544, 1928, 2176, 3080, 5120, 128])
def test_same_bits_on_both_sides_of_the_limit(lib, cols):
    from teletron_amd import ops
    rows, part = (66 << 20) // (2 * cols) + 1, 4 * 211
    g = torch.Generator(device=DEV).manual_seed(cols)
    x, r, dy, ds = (torch.randn(rows, cols, generator=g, device=DEV).to(torch.bfloat16) for _ in range(4))
    a, b, c = (torch.randn(1, cols, generator=g, device=DEV).mul_(0.3).to(torch.bfloat16) for _ in range(3))
    head = 128 if cols % 128 == 0 else 8
    table = torch.randn(rows, head // 2, 2, generator=g, device=DEV)
    st = torch.cuda.current_stream().cuda_stream

    def outputs(n):
        xs, rs, d, e = x[:n], r[:n], dy[:n], ds[:n]
        out = {"adaln": ops.adaln_forward(xs, a, b, EPS), "adaln dx": ops.adaln_backward(d, xs, a, EPS)[0],
               "rms": ops.rmsnorm_forward(xs, c[0], EPS), "rms dx": ops.rmsnorm_backward(d, xs, c[0], EPS)[0],
               "gate": ops.gate_residual_forward(xs, a, rs), "gate dr": ops.gate_residual_backward(d, a, rs)[0]}
        y, xn, inv, dx = torch.empty_like(xs), torch.empty_like(xs), torch.empty(n, device=DEV), torch.empty_like(xs)
        grads = torch.empty(2, cols, dtype=torch.bfloat16, device=DEV)
        ws = torch.empty(lib.tt_adaln_backward_workspace_bytes(n, cols, n), dtype=torch.uint8, device=DEV)
        assert lib.tt_launch_adaln_forward(y.data_ptr(), xn.data_ptr(), xs.data_ptr(), a.data_ptr(), b.data_ptr(), n, cols, EPS,
                                           inv.data_ptr(), st) == 0
        assert lib.tt_launch_adaln_backward(dx.data_ptr(), grads[0].data_ptr(), grads[1].data_ptr(), d.data_ptr(), xn.data_ptr(),
                                            a.data_ptr(), inv.data_ptr(), n, cols, ws.data_ptr(), ws.numel(), st) == 0
        out.update({"saved y": y, "x_norm": xn, "saved dx": dx})
        if cols > 256:
            out["rope"] = ops.rmsnorm_rope_forward(xs, c[0], table[:n], EPS, head)
            out["rope dx"] = ops.rmsnorm_rope_backward(d, xs, c[0], table[:n], EPS, head)[0]
            for name, gate in (("residual", None), ("gated", c)):
                out[name + " s"], out[name + " y"] = ops.residual_norm_forward(xs, rs, gate, a, b, EPS)[:2]
                out[name + " dx"] = ops.residual_norm_backward(d, e, xs, None if gate is None else rs, gate, a, EPS)[0]
        else:
            t = table[:n // 4]
            out["heads"] = ops.rmsnorm_rope_heads_forward(xs.view(1, n // 4, 4, cols), c[0], t, EPS).view(n, cols)
            out["heads dx"] = ops.rmsnorm_rope_heads_backward(d.view(1, n // 4, 4, cols), xs.view(1, n // 4, 4, cols), c[0], t, EPS)[0].view(n, cols)
        return out

    rows = rows // 4 * 4
    large, small = outputs(rows), outputs(part)
    for name in large:
        assert torch.equal(large[name][:part], small[name]), name
