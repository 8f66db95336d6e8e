"""The operators as native autograd nodes against the Python Functions that they stand for: the same bits, and the same
behaviour towards hooks, transforms, freed and changed tensors."""
import threading

import pytest
import torch

from test_gpu_parity import DEV, rand_bf16

pytestmark = pytest.mark.gpu
EPS, B, S, C, H = 1e-6, 2, 37, 1536, 12


def leaf(*shape, seed, scale=1.0, dtype=torch.bfloat16):
    return rand_bf16(*shape, seed=seed, scale=scale).to(DEV).to(dtype).requires_grad_(True)


def cases():
    """name -> (call, inputs): each operator in the forms that models use."""
    import teletron_amd as T
    from teletron_amd import reference_api as R
    x, r = leaf(B, S, C, seed=0), leaf(B, S, C, seed=1)
    mod = [t.detach().requires_grad_(True) for t in rand_bf16(B, 6, C, seed=2, scale=0.3).to(DEV).chunk(6, dim=1)[:3]]
    one, two = leaf(C, seed=3, scale=0.3), leaf(C, seed=4, scale=0.3)
    w32 = leaf(C, seed=5, dtype=torch.float32)
    table = torch.randn(S, C // H // 2, 2, device=DEV, generator=torch.Generator(DEV).manual_seed(6))
    heads = leaf(B, S, H, C // H, seed=7)
    wh = leaf(C // H, seed=8)
    return {
        "adaln": (lambda: T.adaln_modulate(x, mod[0], mod[1], EPS), [x, mod[0], mod[1]]),
        "adaln shared": (lambda: T.AdaLNModelFunction.apply(x, one, two, EPS, C), [x, one, two]),
        "rmsnorm": (lambda: T.RMSNormModelFunction.apply(x, one, EPS, C), [x, one]),
        "rmsnorm fp32": (lambda: T.RMSNormModelFunction.apply(x, w32, EPS, C), [x, w32]),
        "rope": (lambda: T.RMSNormRopeFunction.apply(x, one, table, EPS, H), [x, one]),
        "rope heads": (lambda: T.RMSNormRopeHeadsFunction.apply(heads, wh, table, EPS), [heads, wh]),
        "rope heads view": (lambda: T.RMSNormRopeHeadsFunction.apply(heads.transpose(1, 2), wh, table, EPS), [heads, wh]),
        "gate": (lambda: T.FusedGate()(x, mod[2], r), [x, mod[2], r]),
        "residual": (lambda: T.residual_adaln(x, r, None, mod[0], mod[1], EPS), [x, r, mod[0], mod[1]]),
        "gated residual": (lambda: T.residual_layer_norm(x, r, mod[2], one, two, EPS), [x, r, mod[2], one, two]),
        "saved": (lambda: R.AdaLNModelFunction.apply(x, one, two, EPS, C), [x, one, two]),
    }


NAMES = ["adaln", "adaln shared", "rmsnorm", "rmsnorm fp32", "rope", "rope heads", "rope heads view", "gate", "residual",
         "gated residual", "saved"]


def outs(out):
    return list(out) if isinstance(out, tuple) else [out]


def both(monkeypatch, f):
    """f() through the native nodes, then through the Python Functions."""
    from teletron_amd import ops
    a = f()
    with monkeypatch.context() as m:
        m.setattr(ops, "native", lambda x: None)
        return a, f()


def same(a, b):
    assert len(a) == len(b)
    for p, q in zip(a, b):
        assert (p is None) == (q is None)
        assert p is None or (torch.equal(p, q) and p.dtype == q.dtype and p.stride() == q.stride())


@pytest.mark.parametrize("name", NAMES)
def test_the_native_node_runs(monkeypatch, name):
    """What the tests below compare: the native function takes every one of these calls, with gradients and without."""
    from teletron_amd import functional, ops
    call, _ = cases()[name]
    with monkeypatch.context() as m:
        m.setattr(ops, "native", lambda x: None)
        assert "CppNode" not in outs(call())[0].grad_fn.name()

    def declined(*args):
        raise AssertionError("the native function declined the call")

    monkeypatch.setattr(functional, "_python_apply", declined)
    assert all("CppNode" in t.grad_fn.name() for t in outs(call()))
    with torch.no_grad():
        call()


def test_what_the_graph_shows():
    """Edges, hooks and names of a native node as of any other; a subclass has the Python node with what Python keeps there."""
    import teletron_amd as T
    x, w = leaf(B, S, C, seed=0), leaf(C, seed=1)
    y = T.RMSNormModelFunction.apply(x, w, EPS, C)
    node, seen = y.grad_fn, []
    assert "RMSNormModelFunction" in node.name() and len(node.next_functions) == 2 and node.metadata == {}
    assert not hasattr(node, "saved_tensors")
    node.register_prehook(lambda g: seen.append(g[0].shape))
    node.register_hook(lambda gi, go: seen.append(len(gi)))
    y.sum().backward()
    assert seen == [y.shape, 2]

    class Mine(T.RMSNormModelFunction):
        pass

    z = Mine.apply(x, w, EPS, C)
    assert torch.equal(z, y) and [t.shape for t in z.grad_fn.saved_tensors] == [x.shape, w.shape]


@pytest.mark.parametrize("name", NAMES)
@pytest.mark.parametrize("how", ["dense", "expanded", "misaligned"])
def test_same_bits_for_any_gradient(monkeypatch, name, how):
    def run():
        call, inputs = cases()[name]
        o = outs(call())
        g = []
        for i, t in enumerate(o):
            d = rand_bf16(*t.shape, seed=20 + i).to(DEV)
            if how == "expanded":
                d = d[:, :1].expand(t.shape)
            elif how == "misaligned":
                buf = torch.empty(d.numel() + 3, dtype=d.dtype, device=DEV)
                buf[3:] = d.flatten()
                d = buf[3:].view(d.shape)
            g.append(d)
        return o + list(torch.autograd.grad(o, inputs, g))

    # (a gradient of the view is copied into the rows' order, and so aligned again)
    if how == "misaligned" and name not in ("adaln", "adaln shared", "rmsnorm", "rmsnorm fp32", "rope heads view"):
        with pytest.raises(Exception) as a:
            run()
        from teletron_amd import ops
        monkeypatch.setattr(ops, "native", lambda x: None)
        with pytest.raises(type(a.value)):
            run()
        return
    native, python = both(monkeypatch, run)
    same(native, python)


@pytest.mark.parametrize("name", NAMES)
def test_each_input_alone_and_no_gradients(monkeypatch, name):
    def run():
        results = []
        call, inputs = cases()[name]
        for k in range(len(inputs)):
            for i, t in enumerate(inputs):
                t.requires_grad_(i == k)
            o = outs(call())
            used = [t for t in o if t.requires_grad]
            results += o + list(torch.autograd.grad(used, [inputs[k]], [torch.ones_like(t) for t in used]))
        with torch.no_grad():
            results += outs(call())
        with torch.inference_mode():
            results += outs(call())
        assert not any(t.requires_grad for t in results[-2:])
        return results

    same(*both(monkeypatch, run))


@pytest.mark.parametrize("name", ["residual", "gated residual"])
@pytest.mark.parametrize("which", [0, 1])
def test_one_output_of_the_residual_norm(monkeypatch, name, which):
    def run():
        call, inputs = cases()[name]
        o = call()[which]
        return list(torch.autograd.grad(o, inputs, torch.ones_like(o), allow_unused=True))

    same(*both(monkeypatch, run))


@pytest.mark.parametrize("name", NAMES)
def test_hooks_on_saved_tensors(monkeypatch, name):
    def run():
        call, inputs = cases()[name]
        packed = []

        def pack(t):
            packed.append((tuple(t.shape), t.dtype))
            return t.cpu()

        with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.to(DEV)):
            o = outs(call())
        return packed, o + list(torch.autograd.grad(o, inputs, [torch.ones_like(t) for t in o]))

    (packed, a), (packed_python, b) = both(monkeypatch, run)
    assert packed == packed_python and packed
    same(a, b)

    class Stop(Exception):
        pass

    def stop(t):
        raise Stop

    with pytest.raises(Stop), torch.autograd.graph.saved_tensors_hooks(stop, lambda t: t):
        cases()[name][0]()


def test_saved_view_that_lost_its_strides_is_refused(monkeypatch):
    """Rows are read in the memory order of the saved view, so a hook has to give the strides back."""
    def run():
        call, inputs = cases()["rope heads view"]
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t.contiguous(), lambda t: t):
            o = call()
        with pytest.raises(ValueError, match="tokens in memory order"):
            torch.autograd.grad(o, inputs, torch.ones_like(o))

    both(monkeypatch, run)


@pytest.mark.parametrize("reentrant", [False, True])
@pytest.mark.parametrize("name", NAMES)
def test_checkpointed(monkeypatch, name, reentrant):
    from torch.utils.checkpoint import checkpoint

    def run():
        call, inputs = cases()[name]
        o = outs(checkpoint(lambda *a: call(), *inputs, use_reentrant=reentrant))
        torch.autograd.backward(o, [torch.ones_like(t) for t in o])
        return o + [t.grad for t in inputs]

    same(*both(monkeypatch, run))


def raised(f):
    try:
        f()
    except Exception as e:
        return type(e)
    return None


@pytest.mark.parametrize("name", NAMES)
def test_refusals_are_the_same(monkeypatch, name):
    from torch.autograd import forward_ad
    call, inputs = cases()[name]

    def twice():
        o = outs(call())
        torch.autograd.backward(o, [torch.ones_like(t) for t in o])
        torch.autograd.backward(o, [torch.ones_like(t) for t in o])

    def changed():
        o = outs(call())
        with torch.no_grad():
            for t in inputs:
                t.mul_(1.0)
        torch.autograd.backward(o, [torch.ones_like(t) for t in o])

    def output_changed():
        o = outs(call())
        o[0].mul_(2.0)

    def second_order():
        o = outs(call())
        g = torch.autograd.grad(o, inputs[:1], [torch.ones_like(t) for t in o], create_graph=True)
        g[0].sum().backward()

    def dual():
        import teletron_amd as T
        with forward_ad.dual_level():
            x = forward_ad.make_dual(torch.ones(2, 8, C, device=DEV, dtype=torch.bfloat16), torch.ones(2, 8, C, device=DEV, dtype=torch.bfloat16))
            w = inputs[0].new_ones(C)
            return T.AdaLNModelFunction.apply(x, w, w, EPS, C)

    def vmapped():
        import teletron_amd as T
        w = inputs[0].new_ones(C)
        torch.func.vmap(lambda t: T.RMSNormModelFunction.apply(t, w, EPS, C))(torch.ones(2, 8, C, device=DEV, dtype=torch.bfloat16))

    def functional_grad():
        import teletron_amd as T
        w = inputs[0].new_ones(C)
        torch.func.grad(lambda t: T.RMSNormModelFunction.apply(t, w, EPS, C).float().sum())(torch.ones(8, C, device=DEV, dtype=torch.bfloat16))

    # the residual pair saves its own output and copies of the modulation's slices, so changed inputs are none of its own
    expected = {twice: RuntimeError, changed: None if name == "residual" else RuntimeError,
                output_changed: RuntimeError if name == "rope heads view" else None, second_order: RuntimeError,   # an output that is a view
                dual: NotImplementedError, vmapped: RuntimeError, functional_grad: RuntimeError}
    for f, want in expected.items():
        a, b = both(monkeypatch, lambda: raised(f))
        assert a is b is want, f.__name__


def test_wrong_arguments_are_named_as_before():
    import teletron_amd as T
    x, w = leaf(2, 8, 64, seed=0), leaf(64, seed=1)
    with pytest.raises(ValueError):
        T.AdaLNModelFunction.apply(x, w, w, EPS, 32)
    with pytest.raises(ValueError):
        T.AdaLNModelFunction.apply(x, leaf(1, 8, 64, seed=2), leaf(1, 8, 64, seed=3), EPS, 64)
    with pytest.raises(TypeError):
        T.RMSNormModelFunction.apply(x.float(), w, EPS, 64)
    with pytest.raises(TypeError):
        T.RMSNormModelFunction.apply(x, w, EPS)
    with pytest.raises(ValueError):
        T.RMSNormModelFunction.apply(x.cpu(), w.cpu(), EPS, 64)


def test_subclasses_keep_their_own_forward():
    import teletron_amd as T

    class Mine(T.RMSNormModelFunction):
        @staticmethod
        def forward(ctx, x, weight, epsilon, cols):
            return x.clone()

    x, w = leaf(4, 64, seed=0), leaf(64, seed=1)
    assert torch.equal(Mine.apply(x, w, EPS, 64), x)


def test_threads_and_streams():
    """Passes of several threads, each on a stream of its own, give what one alone gives."""
    want = {n: [t.clone() for t in step(n)] for n in NAMES}
    failed = []

    def work(n):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(10):
                    got = step(n)
                    torch.cuda.current_stream().synchronize()
                    same(got, want[n])
        except BaseException as e:
            failed.append((n, e))

    torch.cuda.synchronize()
    threads = [threading.Thread(target=work, args=(n,)) for n in NAMES]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not failed, failed


def step(name):
    call, inputs = cases()[name]
    o = outs(call())
    return o + list(torch.autograd.grad(o, inputs, [torch.ones_like(t) for t in o]))


@pytest.mark.parametrize("name", NAMES)
def test_compiled(name):
    """torch.compile goes round the operators: the same results as without it."""
    call, inputs = cases()[name]

    def step():
        return [2 * t for t in outs(call())]

    want = step()
    grads = [rand_bf16(*t.shape, seed=20 + i).to(DEV) for i, t in enumerate(want)]
    want += torch.autograd.grad(want, inputs, grads)
    torch._dynamo.reset()
    compiled = torch.compile(step, backend="eager")
    for _ in range(2):
        got = compiled()
        same([*got, *torch.autograd.grad(got, inputs, grads)], want)


@pytest.mark.parametrize("name", NAMES)
def test_compiled_autograd(name):
    """A compiled backward calls the native nodes as they are."""
    call, inputs = cases()[name]
    o = outs(call())
    grads = [rand_bf16(*t.shape, seed=20 + i).to(DEV) for i, t in enumerate(o)]
    want = torch.autograd.grad(o, inputs, grads)
    torch._dynamo.reset()
    o = outs(call())
    with torch._dynamo.compiled_autograd._enable(torch.compile(backend="eager")):
        torch.autograd.backward(o, grads)
    same([t.grad for t in inputs], want)


def test_traced():
    """torch.jit.trace sees the Python class, not a result that it would keep as a constant."""
    import teletron_amd as T
    w = leaf(C, seed=1).detach()
    x, other = (leaf(B, S, C, seed=i).detach() for i in (2, 3))
    traced = torch.jit.trace(lambda t: T.RMSNormModelFunction.apply(t, w, EPS, C), x, check_trace=False)
    assert torch.equal(traced(other), T.RMSNormModelFunction.apply(other, w, EPS, C))
