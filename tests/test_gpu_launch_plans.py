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
