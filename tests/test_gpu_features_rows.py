"""The quadratic feature kernels at the edges of their row pieces and column
blocks: widths that are no whole number of 16-byte pieces (element-wise rows),
one block, several, more than four (two per wave), rows around a 32-row tile,
and the weight gradients' row spans.  Against the oracle at the bounds of
test_gpu_features.py."""
import pytest
import torch

from tests.test_gpu_features import test_quad_features_match_oracle as check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("lead,heads,dim", [((1,), 1, 3), ((31,), 2, 20), ((33,), 1, 130), ((64,), 2, 136),
                                            ((97,), 1, 250), ((700,), 3, 64)])
def test_quad_features_at_row_and_block_edges(lead, heads, dim, dtype):
    check(lead, heads, dim, dtype)
