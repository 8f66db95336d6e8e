"""Parameters as a model holds them: slices of a modulation tensor read in place, fp32 weights, bf16
gradients.  Everything must equal, bit for bit, the same call on dense bf16 parameters with fp32
gradients rounded afterwards, which the other tests hold to the oracle."""
import pytest
import torch

from test_gpu_parity import DEV, rand_bf16

pytestmark = pytest.mark.gpu

# narrow, wide full / masked / ragged / odd rows; 100 and 7 have element-wise kernels only
WIDTHS = [7, 100, 128, 200, 264, 512, 576, 1000, 1001, 1536, 5120]


def modulation(b, cols, how):
    t = rand_bf16(b, 6, cols + 16, seed=cols, scale=0.3).to(DEV)
    if how == "chunks":
        return t[:, :, :cols].contiguous().chunk(6, dim=1)[1:4]
    if how == "offset":                        # rows that start anywhere, an uneven stride
        return [t[:, i:i + 1, 3:3 + cols] for i in (1, 2, 3)]
    return [t[:1, i:i + 1, :cols].expand(b, 1, cols) for i in (1, 2, 3)]


def grads(out, inputs, seed):
    outs = list(out) if isinstance(out, tuple) else [out]
    gs = [rand_bf16(*o.shape, seed=seed + i).to(DEV) for i, o in enumerate(outs)]
    return outs + list(torch.autograd.grad(outs, inputs, gs))


@pytest.mark.parametrize("cols", WIDTHS)
@pytest.mark.parametrize("how", ["chunks", "offset", "expand"])
def test_modulation_slices(cols, how):
    from teletron_amd import functional as T
    b, s = 3, 37
    x, r = (rand_bf16(b, s, cols, seed=i).to(DEV).requires_grad_(True) for i in range(2))
    calls = [lambda p: T.adaln_modulate(x, p[0], p[1])]
    if cols % 8 == 0:
        calls.append(lambda p: T.gate_residual(x, p[2], r))
    if cols % 8 == 0 and cols > 256:
        calls += [lambda p: T.residual_adaln(x, r, p[2], p[0], p[1]), lambda p: T.residual_adaln(x, r, None, p[0], p[1])]
        if how != "offset":                    # a weight vector has to be 16-byte aligned there
            calls.append(lambda p: T.residual_layer_norm(x, r, p[2], p[0][0, 0], p[1][0, 0]))
    for n, call in enumerate(calls):
        results = []
        for dense in (False, True):
            p = [(t.contiguous() if dense else t.detach()).requires_grad_(True) for t in modulation(b, cols, how)]
            used = {0: p[:2], 1: p[2:], 2: p, 3: p[:2], 4: p}[n]
            inputs = [x] + ([r] if n else []) + used
            if not dense:
                with torch.no_grad():          # the same output without anything saved
                    plain = call(p)
            out = call(p)
            if not dense:
                for a, c in zip(plain if isinstance(plain, tuple) else (plain,), out if isinstance(out, tuple) else (out,)):
                    assert torch.equal(a, c)
            results.append(grads(out, inputs, seed=5))
        for a, c in zip(*results):
            assert torch.equal(a, c), (cols, how, n)


@pytest.mark.parametrize("cols", WIDTHS)
def test_fp32_weight_equals_its_bf16_rounding(cols):
    from teletron_amd import functional as T
    x = rand_bf16(2, 41, cols, seed=1).to(DEV).requires_grad_(True)
    w32 = (1 + 0.1 * torch.randn(cols, generator=torch.Generator().manual_seed(3))).to(DEV).requires_grad_(True)
    w16 = w32.detach().to(torch.bfloat16).requires_grad_(True)
    a = grads(T.rms_norm(x, w32), [x, w32], 7)
    b = grads(T.rms_norm(x, w16), [x, w16], 7)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    assert a[2].dtype == torch.float32 and torch.equal(a[2].to(torch.bfloat16), b[2])
    heads = x.detach().reshape(2, 41, 1, cols).expand(2, 41, 3, cols).contiguous().transpose(1, 2)
    assert torch.equal(T.rms_norm(heads, w32), T.rms_norm(heads, w16))


@pytest.mark.parametrize("op", ["rope", "rope_heads"])
def test_bf16_gradients_are_the_fp32_ones_rounded(op):
    from teletron_amd import ops
    s, h, d = 33, 24, 128
    x, dy = (rand_bf16(1, s, h, d, seed=i).to(DEV) for i in range(2))
    table = torch.randn(s, d // 2, 2, generator=torch.Generator().manual_seed(2)).to(DEV)
    if op == "rope":
        w, args = rand_bf16(h * d, seed=3).to(DEV), (1e-6, d)
        x, dy, fn = x.flatten(2), dy.flatten(2), ops.rmsnorm_rope_backward
    else:
        w, args, fn = rand_bf16(d, seed=3).to(DEV), (1e-6,), ops.rmsnorm_rope_heads_backward
    (dx, g), (dx16, g16) = fn(dy, x, w, table, *args), fn(dy, x, w, table, *args, dtype=torch.bfloat16)
    assert torch.equal(dx, dx16) and g.dtype == torch.float32 and torch.equal(g.to(torch.bfloat16), g16)


@pytest.mark.parametrize("cols", [7, 100, 128, 1000, 1001, 1536])
def test_native_calls_equal_the_python_ones(cols, monkeypatch):
    """ops.native() covers the ordinary calls; what it declines, and other tensor classes, take ops.py."""
    from teletron_amd import functional as T, ops

    class Tagged(torch.Tensor):
        pass

    x, r = (rand_bf16(2, 29, cols, seed=i).to(DEV).requires_grad_(True) for i in range(2))
    assert ops.native(x) is not None and ops.native(x.detach().as_subclass(Tagged)) is None and ops.native(x.cpu()) is None
    assert ops.native(x).adaln_forward(x.float(), x[:, :1], x[:, :1], 1e-6, False) is None
    p = [t.detach().requires_grad_(True) for t in modulation(2, cols, "chunks")]
    w = p[0].detach()[0, 0].clone().requires_grad_(True)
    calls = [(lambda: T.adaln_modulate(x, p[0], p[1]), [x, p[0], p[1]]), (lambda: T.rms_norm(x, w), [x, w])]
    if cols % 8 == 0:
        calls.append((lambda: T.gate_residual(x, p[2], r), [x, p[2], r]))
        table = torch.randn(29, cols // 2, 2, device=DEV)
        heads = x.detach().reshape(2, 29, 1, cols).expand(2, 29, 3, cols).contiguous().requires_grad_(True)
        if cols <= 256:
            calls.append((lambda: T.RMSNormRopeHeadsFunction.apply(heads.transpose(1, 2), w, table, 1e-6), [heads, w]))
    if cols == 1536:
        calls += [(lambda: T.residual_adaln(x, r, p[2], p[0], p[1]), [x, r, *p]),
                  (lambda: T.RMSNormRopeFunction.apply(x, w, table[:, :64].contiguous(), 1e-6, 12), [x, w])]
    native = [grads(call(), inputs, 3) for call, inputs in calls]
    monkeypatch.setattr(ops, "native", lambda x: None)
    for (call, inputs), got in zip(calls, native):
        for a, b in zip(got, grads(call(), inputs, 3)):
            assert torch.equal(a, b)


def test_operators_run_without_the_native_module(monkeypatch):
    """As after a build of the C ABI alone: the same bits through ops.py."""
    import importlib.util
    from teletron_amd import functional as T, ops
    x = rand_bf16(2, 29, 1536, seed=1).to(DEV).requires_grad_(True)
    w = rand_bf16(1536, seed=2).to(DEV).requires_grad_(True)
    want = grads(T.rms_norm(x, w), [x, w], 3) + grads(T.adaln_modulate(x, w, w), [x, w], 3)
    find = importlib.util.find_spec
    monkeypatch.setattr(importlib.util, "find_spec", lambda name, *a: None if name.endswith("native_ops") else find(name, *a))
    monkeypatch.setitem(__import__("sys").modules, "teletron_amd.native_ops", None)      # and importing it would raise
    monkeypatch.delattr("teletron_amd.native_ops")
    monkeypatch.setattr(ops, "_native", None)
    got = grads(T.rms_norm(x, w), [x, w], 3) + grads(T.adaln_modulate(x, w, w), [x, w], 3)
    assert ops.native(x) is None
    ops.clear_workspaces()
    for a, b in zip(got, want):
        assert torch.equal(a, b)
