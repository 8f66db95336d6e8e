"""Widths whose workgroups hold more row groups than the others of their kernels: rows that are no multiple of a tile,
one row, several tiles a workgroup."""
import pytest
import torch

from test_gpu_parity import DEV, check_adaln, check_rmsnorm, rand_bf16

pytestmark = pytest.mark.gpu


# 3, 4 and 6 waves of two packs: full rows and ones with idle lanes
@pytest.mark.parametrize("heads", [17, 20, 24, 25, 32, 41, 48])
@pytest.mark.parametrize("b,s", [(1, 1), (3, 7), (2, 1601)])
def test_rotary_backward(heads, b, s):
    from oracle import norm_oracle as O
    from teletron_amd import ops
    from test_gpu_parity import assert_bf16_close, assert_grad_close
    c = heads * 128
    x, dy = rand_bf16(b, s, c, seed=heads), rand_bf16(b, s, c, seed=heads + 1)
    w = rand_bf16(c, seed=heads + 2, scale=0.1, offset=1.0)
    ang = 3.0 * torch.randn(s, 64, generator=torch.Generator().manual_seed(s))
    table = torch.stack([ang.cos(), ang.sin()], dim=-1)
    dx, dw = ops.rmsnorm_rope_backward(dy.to(DEV), x.to(DEV), w.to(DEV), table.to(DEV), 1e-6, 128)
    dxo, dwo = O.rmsnorm_rope_backward(dy, x, w, table, 1e-6, 128)
    assert_bf16_close(dx, dxo, "dx")
    assert_grad_close(dw, dwo, b * s, "dweight")


# ragged rows: the shortest and the longest of the variants of 2, 3 and 4 waves of one pack, 3, 4 and 5 of two
@pytest.mark.parametrize("cols", [520, 1000, 1032, 1528, 1544, 2040, 2056, 3064, 3080, 4088, 4104, 5112])
@pytest.mark.parametrize("nb,rpb", [(1, 1), (2, 31), (1, 1901)])
def test_ragged_rows(cols, nb, rpb):
    from test_gpu_gate import test_gate_residual_shapes as check_gate
    from test_gpu_resnorm import run_case as check_residual
    x, dy = rand_bf16(nb, rpb, cols, seed=cols), rand_bf16(nb, rpb, cols, seed=cols + 1)
    p = [rand_bf16(nb, 1, cols, seed=cols + 2 + i, scale=0.2) for i in range(2)]
    check_adaln(x, p[0], p[1], dy, 1e-6, nb, f"cols {cols}")
    check_rmsnorm(x, 1 + p[0][0, 0], dy, 1e-6, f"cols {cols}")
    check_gate(cols, nb, rpb)
    for gated in (False, True):
        check_residual(cols, nb, rpb, gated, affine=False)


@pytest.mark.parametrize("cols", [1000, 1992])
def test_same_rows_with_batches_that_divide_the_cus_badly(cols):
    """Beyond the caches their workgroups hold fewer row groups: the same bits a row as with one batch."""
    from teletron_amd import ops
    nb = 140
    rpb = (70 << 20) // (2 * cols * nb) + 1
    x = torch.randn(nb * rpb, cols, generator=torch.Generator(DEV).manual_seed(cols), device=DEV).to(torch.bfloat16)
    a, b = (rand_bf16(1, cols, seed=i, scale=0.3).to(DEV) for i in range(2))
    one = ops.adaln_forward(x, a, b, 1e-6)
    assert torch.equal(ops.adaln_forward(x, a.expand(nb, cols).contiguous(), b.expand(nb, cols).contiguous(), 1e-6), one)
