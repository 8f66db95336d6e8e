"""Head counts whose rows a wave takes token by token (3 to 6 loads of 4 or 8 rows), beside ones that it
does not, at the edges of a tile.  Oracle and tolerances as in test_gpu_rope.py."""
import pytest

from test_gpu_rope import test_rmsnorm_rope_heads_shapes as check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads", [4, 12, 16, 20, 32, 36, 40, 48, 60])
@pytest.mark.parametrize("hd", [40, 64, 72, 128])
@pytest.mark.parametrize("b,s", [(1, 1), (2, 53)])
def test_token_mode_head_counts(heads, hd, b, s):
    check(b, s, heads, hd)
