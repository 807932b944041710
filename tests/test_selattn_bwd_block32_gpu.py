"""GPU: selected attention backward with blocks of 32 (passes of 32 gathered rows, of 64 at head_dim 64) at the edges of a pass:
blocks with fewer rows than one, exactly one, one more, and blocks that several work-groups share, against the CPU oracle."""
import pytest
import torch

from test_selattn_bwd_gpu import test_bwd_matches_oracle as _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,dtype", [(64, torch.float16), (128, torch.bfloat16), (256, torch.float16)])
@pytest.mark.parametrize("cu,hq,hkv,t", [
    ([0, 1, 32, 65], 2, 2, 4),         # sequences of 1, 31 and 33 tokens
    ([0, 64], 1, 1, 1),                # every block has the rows of its own queries: one pass
    ([0, 650], 3, 1, 8),               # three heads to a group: passes that begin inside a query
    ([0, 2500], 8, 1, 16),             # block 0 is everybody's
])
def test_blocks_of_32(dev, cu, hq, hkv, t, d, dtype):
    _check(dev, cu, hq, hkv, d, 32, t, dtype, 0.5)
