"""Head counts whose rows a wave takes token by token (3 to 6 loads of 4 or 8 rows), beside ones that it
does not, at the edges of a tile.  Oracle and tolerances as in test_gpu_rope.py.  Tensors that fit the caches (64 MiB) look every
row up in backward, and in forward unless there is a tile for every CU; the larger ones below run
token by token both ways, over several tiles a workgroup and past the wrap of the positions."""
import pytest
import torch

from test_gpu_configs import whole_tensor_check
from test_gpu_parity import DEV, assert_grad_close
from test_gpu_rope import test_rmsnorm_rope_heads_shapes as check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads", [4, 12, 16, 20, 32, 36, 40, 48, 60])
@pytest.mark.parametrize("hd", [40, 64, 72, 128])
@pytest.mark.parametrize("b,s", [(1, 1), (2, 53)])
def test_token_mode_head_counts(heads, hd, b, s):
    check(b, s, heads, hd)


# six, four and three loads a wave, rows of 16 and of 8 lanes, with every lane in use and without; 40 heads: per row
@pytest.mark.parametrize("mib", [20, 68])
@pytest.mark.parametrize("heads,hd", [(h, d) for d in (128, 72) for h in (12, 16, 24, 40, 48, 60)] +
                         [(h, d) for d in (64, 40) for h in (24, 32, 48)])
def test_token_mode_over_many_tiles(heads, hd, mib):
    """Every element against torch fp32 on the GPU, the weight gradient against fp64 sums."""
    from teletron_amd import ops
    b, eps = 2, 1e-6
    s = (mib << 20) // (2 * b * heads * hd) + 1
    g = torch.Generator(device=DEV).manual_seed(heads + hd)
    x, dy = (torch.randn(b, s, heads, hd, generator=g, device=DEV).to(torch.bfloat16) for _ in range(2))
    assert (x.numel() * 2 >= 64 << 20) == (mib > 64)
    w = (1 + 0.1 * torch.randn(hd, generator=g, device=DEV)).to(torch.bfloat16)
    ang = 3.0 * torch.randn(s, hd // 2, generator=g, device=DEV)
    table = torch.stack([ang.cos(), ang.sin()], dim=-1).contiguous()
    y = ops.rmsnorm_rope_heads_forward(x, w, table, eps)
    dx, dw = ops.rmsnorm_rope_heads_backward(dy, x, w, table, eps)
    fc = torch.view_as_complex(table)[None, :, None]                       # [1, S, 1, D/2]

    def rot(t, f):
        return torch.view_as_real(torch.view_as_complex(t.unflatten(-1, (-1, 2)).contiguous()) * f).flatten(-2)
    xf = x.float()
    rstd = torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + eps)
    xh, dn = xf * rstd, rot(dy.float(), fc.conj())
    gg = dn * w.float()
    refs = {"y": (y, rot(xh * w.float(), fc)), "dx": (dx, rstd * (gg - xh * (gg * xh).mean(-1, keepdim=True)))}
    for got, ref in refs.values():
        ref = ref.reshape(b * s, heads * hd)
        whole_tensor_check(got.reshape(b * s, heads * hd), lambda r0, r1: ref[r0:r1], 8192)
    assert_grad_close(dw, (dn.double() * xh.double()).sum((0, 1, 2)).cpu(), b * s * heads, "dweight")
