"""The quadratic feature-map kernels (gpa_amd/csrc/quad_features.hip) built for
the host under AddressSanitizer (tests/host_emu/) and compared on the CPU with
the oracle's restatement of the reference's map (oracle.reference
.quadratic_features, src/gpa/features.py:17-25): forward output and the
gradients of x and of every parameter, float32 (1e-5 / 1e-4) and bfloat16
(2e-2), for widths below, at and above one 32-column block (8, 32, 40, 128,
256), partial row tiles and a zero row.  Every access of the kernels is
bounds-checked here before they run on a GPU.  Parameters that do not fit x's
heads, width or device are refused before any kernel runs.
"""
import math

import pytest
import torch

from gpa_amd import features
from gpa_amd.module import QuadraticFeatures
from oracle import reference as ref
from tests.host_emu import harness


@pytest.fixture
def host(host_runner, tmp_path, monkeypatch):
    lib = harness.HostLib(host_runner, str(tmp_path))
    harness.use_host(monkeypatch, lib)
    return lib


def _rel(a, b):
    a, b = a.detach().double(), b.detach().double()
    return ((a - b).norm() / max(b.norm().item(), 1e-30)).item()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("rows,heads,dim", [(37, 2, 8), (32, 1, 32), (65, 2, 40), (40, 1, 128), (33, 1, 256)])
def test_quad_features_match_oracle(host, rows, heads, dim, dtype):
    torch.manual_seed(rows + dim)
    fm = QuadraticFeatures(heads, dim)
    with torch.no_grad():
        fm.gain_raw.normal_(0, .5)
    x = torch.randn(rows, heads, dim).to(dtype)
    x[3] = 0  # a zero row: both normalisations at their floors
    w = torch.randn(rows, heads, dim)

    def run(fn):
        xx = x.clone().requires_grad_()
        fm.zero_grad(set_to_none=True)
        y = fn(xx)
        (y.float() * w).sum().backward()
        return [y, xx.grad, fm.left.grad, fm.right.grad, fm.gain_raw.grad]

    def kernel(xx):
        gain = 2 * fm.gain_raw.sigmoid() * math.sqrt(dim)
        return features._QuadFeatures.apply(xx, fm.left, fm.right, gain)

    got = run(kernel)
    want = run(lambda xx: ref.quadratic_features(fm, xx))
    tol = (1e-5, 1e-4) if dtype == torch.float32 else (2e-2, 3e-2)
    for i, (name, a, r) in enumerate(zip(("out", "dx", "dleft", "dright", "dgain"), got, want)):
        assert _rel(a, r) < tol[min(i, 1)], (name, _rel(a, r))


@pytest.mark.parametrize("wrong", [dict(right=(1, 8, 8)), dict(left=(1, 8, 8)), dict(left=(1, 8, 8), right=(1, 8, 8)),
                                   dict(right=(2, 8, 4)), dict(left=(2, 4, 8)), dict(right=(2, 64)),
                                   dict(left=(3, 8, 8), right=(3, 8, 8)), dict(gain=(1,))], ids=str)
def test_quad_features_refuse_parameters_of_other_shapes(host, wrong):
    """The kernels address the matrices and the gain by x's heads and width:
    parameters that hold fewer values would be read past their end."""
    from gpa_amd import _lib
    shapes = {**dict(left=(2, 8, 8), right=(2, 8, 8), gain=(2,)), **wrong}
    x = torch.randn(5, 2, 8)
    with pytest.raises(_lib.HipBackendError, match="quadratic features"):
        features._QuadFeatures.apply(x, *(torch.randn(shapes[n]) for n in ("left", "right", "gain")))


@pytest.mark.parametrize("name", ["left", "right", "gain"])
def test_quad_features_refuse_parameters_on_another_device(host, name):
    from gpa_amd import _lib
    params = dict(left=torch.randn(2, 8, 8), right=torch.randn(2, 8, 8), gain=torch.randn(2))
    params[name] = params[name].to("meta")
    with pytest.raises(_lib.HipBackendError, match="quadratic features"):
        features._QuadFeatures.apply(torch.randn(5, 2, 8), *params.values())


@pytest.mark.parametrize("dim", [16, 130])
def test_quad_features_round_every_quotient(host, dim):
    """out = unit(x)/|unit(x)| |x| with zero weight matrices and two nonzero elements
    a row, in two lanes' sums, so that no sum depends on an order: bit for bit, each
    quotient rounded by itself (a factor |x|/|unit(x)| per row rounds otherwise)."""
    gen, at = torch.Generator().manual_seed(dim), [3, 12]
    x, want = torch.zeros(40, 1, dim), torch.zeros(40, 1, dim)
    pair = torch.randn(40, 1, 2, generator=gen)
    ss = (pair * pair).sum(-1, keepdim=True)
    u = pair / ss.sqrt()
    x[..., at] = pair
    want[..., at] = u / (u * u).sum(-1, keepdim=True).sqrt() * (ss + 1e-12).sqrt()
    zero = torch.zeros(1, dim, dim)
    assert torch.equal(features._QuadFeatures.apply(x, zero, zero, torch.ones(1)), want)
