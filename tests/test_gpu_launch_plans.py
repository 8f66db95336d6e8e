"""Launch plans that the figures beside the kernels rest on, as the size queries and workspaces show them."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cols", [520, 1000, 1024, 1032, 1536])
@pytest.mark.parametrize("rows", [4096, 20000])
def test_residual_norm_backward_keeps_one_workgroup_a_cu(lib, rows, cols):
    """Two and three waves a row: with fewer registers a second workgroup would fit, whose partial sums cost
    more than it gives."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert lib.tt_residual_norm_backward_workspace_bytes(rows, cols, rows, 0) == cus * 2 * cols * 4


def partials_a_batch(lib, rows, cols, nb, op="adaln"):
    """Workgroups a batch that the backward of a norm launches, and the size query's answer."""
    import ctypes
    x, dy, dx = (torch.ones(rows, cols, dtype=torch.bfloat16, device="cuda:0") for _ in range(3))
    p = torch.ones(nb, cols, dtype=torch.bfloat16, device="cuda:0")
    shape = [rows, cols, rows // nb] if op == "adaln" else [rows, cols]
    need = getattr(lib, f"tt_{op}_backward_workspace_bytes")(*shape)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda:0")
    n = ctypes.c_int(0)
    args = [dx.data_ptr(), dy.data_ptr(), x.data_ptr(), p.data_ptr(), ws.data_ptr(), need, ctypes.byref(n)]
    assert getattr(lib, f"tt_{op}_backward_partials")(*args, *shape, 1e-6, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    return n.value, need


@pytest.mark.parametrize("rows,cols,nb", [(2000, 3072, 1), (9000, 3072, 3), (1200, 5128, 1), (3000, 1536, 2), (4300, 3072, 43), (86 * 34, 2696, 86),
                                          (60 * 200, 1536, 200)])
def test_cached_backward_of_wide_rows_runs_one_workgroup_a_cu(lib, rows, cols, nb):
    """... and no more than the size query's answer, at most a third of the CUs going without."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    n, need = partials_a_batch(lib, rows, cols, nb)
    assert n == cus // nb and n * nb * 3 >= cus * 2 and n * nb * 2 * cols * 4 <= need


@pytest.mark.parametrize("nb", [129, 140, 168, 300])
def test_batches_that_divide_the_cus_badly_keep_every_cu(lib, nb):
    """One workgroup a CU in whole workgroups a batch would leave over a third of the CUs without one."""
    cus, cols, rpb = torch.cuda.get_device_properties(0).multi_processor_count, 2312, 20
    assert cus // nb * nb * 3 < cus * 2
    n, need = partials_a_batch(lib, rpb * nb, cols, nb)
    assert n * nb * 3 >= cus * 2 and n * nb * 2 * cols * 4 <= need


@pytest.mark.parametrize("rows,cols,capped", [(19660, 640, False), (19660, 648, False), (6009, 1664, False), (2403, 1664, True), (5208, 1920, True),
                                              (6475, 1544, False), (6510, 1536, True)])
def test_rows_with_idle_lanes_keep_their_workgroups(lib, rows, cols, capped):
    """Over a quarter of the lanes without a pack, or over a sixteenth beyond 12 MiB: as many workgroups as fit a CU."""
    n, _ = partials_a_batch(lib, rows, cols, 1, "rmsnorm")
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert n == cus if capped else n > cus
