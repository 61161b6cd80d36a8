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


@pytest.mark.parametrize("rows,heads,dim", [(4097, 2, 128), (700, 3, 64), (9000, 1, 200), (30, 2, 40)])
def test_weight_gradients_repeat(rows, heads, dim):
    """The bf16 weight gradients add their row spans (1 to 256 of them here) in
    a fixed order: equal calls give equal bits."""
    from gpa_amd.module import QuadraticFeatures
    torch.manual_seed(rows)
    fm = QuadraticFeatures(heads, dim).cuda()
    x = torch.randn(rows, heads, dim, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    w = torch.randn(rows, heads, dim, device="cuda", dtype=torch.bfloat16)
    grads = [torch.autograd.grad(fm(x), (x, *fm.parameters()), w) for _ in range(6)]
    for again in grads[1:]:
        assert all(torch.equal(a, b) for a, b in zip(grads[0], again))


def test_quad_features_of_many_heads():
    """Heads up to the launch limit of 65535 (one workgroup row per head): the
    weight layouts, which take two matrices per head, included.  Forward against
    the oracle at test_gpu_features.py's float32 bound."""
    from gpa_amd.module import QuadraticFeatures
    from oracle import reference as ref
    from tests.test_gpu_features import _rel
    heads, dim = 65535, 2
    torch.manual_seed(0)
    many = QuadraticFeatures(1, dim)
    many.left, many.right = (torch.nn.Parameter(torch.randn(heads, dim, dim)) for _ in range(2))
    many.gain_raw = torch.nn.Parameter(torch.randn(heads))
    x = torch.randn(3, heads, dim)
    with torch.no_grad():
        want = ref.quadratic_features(many, x)
        got = many.cuda()(x.cuda())
    assert _rel(got, want) < 1e-5
