"""Two host threads that call a backward operator on the same stream share its workspace: the kernels of
one call have to be queued before those of the other."""
import contextlib
import ctypes
import threading
import time
import types

import pytest
import torch


def run_threads(work, n=2):
    errors = []

    def body(i):
        try:
            work(i)
        except BaseException as e:
            errors.append(e)
    threads = [threading.Thread(target=body, args=(i,)) for i in range(n)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    if errors:
        raise errors[0]


def test_a_call_has_the_workspace_to_itself_until_its_launches_are_queued(monkeypatch):
    """The C ABI call, with the GIL released, stands in for kernel and reduction: what it wrote into the workspace
    first must be there at its end, while another thread makes the same call."""
    from teletron_amd import cabi, ops
    monkeypatch.setattr(ops, "_check_act", lambda name, t, cols: t)
    monkeypatch.setattr(ops, "_check_param", lambda name, p, ref, cols: p)
    monkeypatch.setattr(ops, "_stream", lambda t: 7)
    monkeypatch.setattr(torch.cuda, "device", lambda d: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(cabi, "load", lambda: types.SimpleNamespace(tt_gate_residual_backward_workspace_bytes=lambda *a: 64))
    clashes = []

    def call(name, *args):
        ws = ctypes.c_int64.from_address(args[6])
        ws.value = me = threading.get_ident()
        time.sleep(0.01)
        if ws.value != me:
            clashes.append(name)
    monkeypatch.setattr(cabi, "call", call)
    x = torch.zeros(4, 8)

    def work(i):
        for _ in range(5):
            ops.gate_residual_backward(x, x[:1], x)
    try:
        run_threads(work)
    finally:
        ops.clear_workspaces()
    assert not clashes


@pytest.mark.gpu
@pytest.mark.parametrize("path", ["native", "ops", "dispatcher"])
def test_two_threads_on_one_stream_get_their_own_gradients(path):
    from teletron_amd import fused_rmsnorm, ops  # noqa: F401  (registers the dispatcher names)
    dev, rows, cols, eps = "cuda:0", 512, 1024, 1e-6
    g = torch.Generator(device=dev).manual_seed(0)
    sets = [[torch.randn(rows, cols, generator=g, device=dev).to(torch.bfloat16) for _ in range(2)] for _ in range(2)]
    w = torch.ones(cols, device=dev, dtype=torch.bfloat16)

    def call(x, dy):
        if path == "native":
            return ops.native(x).rmsnorm_backward(dy, x, w, None, eps, 0, 0, False, (cols,))[1]
        if path == "ops":
            return ops.rmsnorm_backward(dy, x, w, eps)[1]
        dx, dw, inv = torch.empty_like(x), torch.empty_like(w), torch.ones(rows, device=dev)
        torch.ops.Fused_RMSNorm.torch_launch_rms_backward(dx, dw, dy, x, w, inv, rows, cols)
        return dw

    want = [call(*s) for s in sets]
    assert not torch.equal(*want)

    def work(i):
        got = [call(*sets[i]) for _ in range(300)]
        torch.cuda.synchronize()
        assert all(torch.equal(t, want[i]) for t in got)
    run_threads(work)
