"""The bf16 chunk preparation (gdn_prep_frag) where its loads and tiles have
edges: rows on and off 16-byte boundaries (16-byte and element-wise loads),
key widths below, between and at the 64/128/256 classes, value widths with a
partial 8-value piece, a partial 32-column strip, two 128-value slices, and
above 256 (saved rows in float32).  Rows that start off a boundary hold the
same values, so every result has the same bits; against the recurrence the
bound is the scan tests' 2e-2 (a bf16 read rounds at 2^-9)."""
import pytest
import torch

from tests.test_gpu_gdn_scan import DEV, _inputs, _oracle_segments, _oracle_segments_autograd, _rel

pytestmark = pytest.mark.gpu

CASES = [(1, 16, 8, 64, 0), (70, 48, 20, 64, 5), (129, 64, 33, 64, 63), (66, 80, 96, 64, 0), (65, 128, 256, 64, 0),
         (40, 128, 130, 16, 3), (70, 192, 128, 64, 17), (64, 256, 8, 64, 0), (65, 128, 264, 64, 1)]


def _off_boundary(x):
    """The same values in rows that start 2 bytes past a 16-byte boundary."""
    wide = torch.zeros(*x.shape[:-1], x.shape[-1] + 9, dtype=x.dtype, device=x.device)
    wide[..., 1:x.shape[-1] + 1] = x
    return wide[..., 1:x.shape[-1] + 1]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "T{}K{}V{}C{}o{}".format(*c))
def test_prep_rows_on_and_off_boundaries(case):
    from gpa_amd.ops import gdn_scan_hip
    t, kd, vd, chunk, offset = case
    q, k, v, g, beta, s0 = _inputs(2, t, 2, kd, vd, torch.bfloat16, seed=31)
    args = [x.to(DEV) for x in (q, k, v)], [x.to(DEV) for x in (g, beta, s0)]
    got = gdn_scan_hip(*args[0], *args[1], chunk=chunk, offset=offset)
    moved = gdn_scan_hip(*(_off_boundary(x) for x in args[0]), *args[1], chunk=chunk, offset=offset)
    assert all(torch.equal(a, b) for a, b in zip(got, moved))
    errs = [_rel(a, b) for a, b in zip(got, _oracle_segments(q, k, v, g, beta, s0, chunk, offset))]
    print(case, errs)
    assert max(errs) < 2e-2, errs


@pytest.mark.parametrize("with_q", [True, False], ids=["read", "noread"])
@pytest.mark.parametrize("case", [c for c in CASES if c[1] * c[2] <= 128 * 256], ids=lambda c: "T{}K{}V{}C{}o{}".format(*c))
def test_chunk_backward_rows_on_and_off_boundaries(case, with_q):
    """The fragment chunk backward (gdn_chunk_bwd_frag; aligned rows, V % 8 == 0)
    and the one it leaves to other rows, at the same edges: partial rounds of 32
    values, one and two row tiles, partial key tiles."""
    from gpa_amd.ops import gdn_scan_hip
    t, kd, vd, chunk, offset = case
    inputs = _inputs(2, t, 2, kd, vd, torch.bfloat16, seed=37, q=with_q)
    gen = torch.Generator().manual_seed(3)
    refs = [x.double().requires_grad_() if x is not None else None for x in inputs]
    want = _oracle_segments_autograd(refs[:3], *refs[3:], chunk, offset)
    w = [torch.randn(x.shape, generator=gen).to(torch.bfloat16) for x in want]
    pick = (0, 1, 2) if with_q else (1, 2)
    dr = torch.autograd.grad([want[i] for i in pick], [x for x in refs if x is not None], [w[i].double() for i in pick])
    for move in (lambda x: x, _off_boundary):
        leaves = [x.to(DEV).requires_grad_() if x is not None else None for x in inputs]
        args = [move(x) if x is not None else None for x in leaves[:3]] + leaves[3:]
        got = gdn_scan_hip(*args, chunk=chunk, offset=offset)
        dg = torch.autograd.grad([got[i] for i in pick], [x for x in leaves if x is not None],
                                 [w[i].to(DEV, got[i].dtype) for i in pick])
        errs = [_rel(a, b) for a, b in zip(dg, dr)]
        print(case, with_q, errs)
        assert max(errs) < 2e-2, errs
