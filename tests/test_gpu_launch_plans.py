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


@pytest.mark.parametrize("rows,cols,nb", [(2000, 3072, 1), (9000, 3072, 3), (1200, 5128, 1), (3000, 1536, 2), (600, 512, 600)])
def test_cached_backward_of_wide_rows_runs_one_workgroup_a_cu(lib, rows, cols, nb):
    """... and no more than the size query's answer; rows with over a quarter of their lanes idle keep theirs."""
    import ctypes
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    x, dy, dx = (torch.ones(rows, cols, dtype=torch.bfloat16, device="cuda:0") for _ in range(3))
    p = torch.ones(nb, cols, dtype=torch.bfloat16, device="cuda:0")
    need = lib.tt_adaln_backward_workspace_bytes(rows, cols, rows // nb)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda:0")
    n = ctypes.c_int(0)
    args = [dx.data_ptr(), dy.data_ptr(), x.data_ptr(), p.data_ptr(), ws.data_ptr()]
    tail = [rows, cols, rows // nb, 1e-6, torch.cuda.current_stream().cuda_stream]
    assert lib.tt_adaln_backward_partials(*args, need, ctypes.byref(n), *tail) == 0
    torch.cuda.synchronize()
    assert 1 <= n.value <= max(1, cus // nb) and n.value * nb * 2 * cols * 4 <= need
