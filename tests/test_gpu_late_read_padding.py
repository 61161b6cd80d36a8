"""A late read (gdn_scan_deferred) whose keys end inside a 32-key tile: the
padding of its query fragments is zero whatever the memory held, so that the
scan backward, which multiplies whole tiles, gives the gradients of the scan
with the read built in.  New memory is filled with NaN for the test.  Bound:
both round the same products to bf16, at 2^-9 each, so 2e-2 as for the scan."""
import pytest
import torch

from tests.test_gpu_gdn_scan import DEV, _inputs, _rel

pytestmark = pytest.mark.gpu


@pytest.fixture
def nan_memory():
    was = torch.are_deterministic_algorithms_enabled(), torch.is_deterministic_algorithms_warn_only_enabled()
    torch.use_deterministic_algorithms(True, warn_only=True)  # new tensors start as NaN
    yield
    torch.use_deterministic_algorithms(was[0], warn_only=was[1])


@pytest.mark.parametrize("kd", [16, 48, 80, 144, 64])
def test_late_read_in_new_memory(nan_memory, kd):
    from gpa_amd.ops import gdn_scan_deferred, gdn_scan_hip
    inputs = _inputs(2, 21, 2, kd, 24, torch.bfloat16, seed=5)
    gen = torch.Generator().manual_seed(3)
    res = []
    for late in (False, True):
        leaves = [x.to(DEV).requires_grad_() for x in inputs]
        q, rest = leaves[0], leaves[1:]
        if late:
            states, final, read = gdn_scan_deferred(*rest, chunk=8, offset=3)
            out = read(q)
        else:
            out, states, final = gdn_scan_hip(q, *rest, chunk=8, offset=3)
        w = [torch.randn(x.shape, generator=gen.manual_seed(3)).to(DEV, x.dtype) for x in (out, states, final)]
        res.append((out, *torch.autograd.grad((out, states, final), leaves, w)))
    errs = [_rel(a, b) for a, b in zip(res[1], res[0])]
    print(kd, errs)
    assert all(e < 2e-2 for e in errs), errs  # (a NaN fails)


@pytest.mark.parametrize("kd,vd", [(48, 24), (128, 128), (256, 64)])
def test_late_read_has_the_bits_of_the_read_built_in(kd, vd):
    """Queries are normalised by two kernels (the scan's preparation and, for a
    late read, gdn_prep_q) that sum a row's squares alike: the outputs are equal."""
    from gpa_amd.ops import gdn_scan_deferred, gdn_scan_hip
    q, *rest = (x.to(DEV) for x in _inputs(2, 700, 4, kd, vd, torch.bfloat16, seed=8))
    out, states, final = gdn_scan_hip(q, *rest, chunk=64, offset=0)
    late_states, late_final, read = gdn_scan_deferred(*rest, chunk=64, offset=0)
    assert torch.equal(states, late_states) and torch.equal(final, late_final)
    assert torch.equal(out, read(q))
