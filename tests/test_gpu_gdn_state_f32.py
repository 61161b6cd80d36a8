"""The float32 state recurrences (gdn_state_fwd / gdn_state_bwd, 16 state
columns per workgroup, key rows split over four waves) at the edges of their
tiles: key widths at and around the 64/128/256 classes, whole and partial
16-wide key groups, one and partial 16-column tiles, chunks of few rows.
Compared with the oracle's recurrence in float64 at 1e-5: sums of at most 256
float32 products, each scaled by e^g <= 1, over a chain of at most 4 chunks."""
import pytest
import torch

from tests.test_gpu_gdn_scan import DEV, _inputs, _oracle_segments_autograd, _rel

pytestmark = pytest.mark.gpu

# (T, K, V, chunk, offset)
CASES = [(1, 16, 16, 64, 0), (70, 80, 17, 64, 5), (9, 64, 1, 3, 1), (130, 144, 33, 64, 63), (20, 256, 15, 8, 3),
         (67, 18, 16, 32, 0), (40, 130, 5, 16, 2), (33, 68, 48, 64, 0)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "T{}K{}V{}C{}o{}".format(*c))
def test_float32_state_matches_recurrence(case):
    from gpa_amd.ops import gdn_scan_hip
    t, kd, vd, chunk, offset = case
    inputs = _inputs(2, t, 2, kd, vd, torch.float32, seed=21)
    leaves = [x.to(DEV).requires_grad_() for x in inputs]
    refs = [x.double().requires_grad_() for x in inputs]
    got = gdn_scan_hip(*leaves, chunk=chunk, offset=offset)
    want = _oracle_segments_autograd(refs[:3], *refs[3:], chunk, offset)
    gen = torch.Generator().manual_seed(3)
    grads = [torch.randn(x.shape, generator=gen, dtype=torch.float64) for x in want]
    dg = torch.autograd.grad(got, leaves, [x.to(DEV, torch.float32) for x in grads])
    dr = torch.autograd.grad(want, refs, [x.float().double() for x in grads])
    errs = [_rel(a, b) for a, b in zip((*got, *dg), (*want, *dr))]
    print(case, errs)
    assert max(errs) < 1e-5, errs


def telescoping(scan, device, kd=64):
    """(final state's rows, last value) of a float32 scan of 150 tokens whose
    keys all point one way and whose writes are full: S_t = k v_t^T."""
    gen = torch.Generator().manual_seed(4)
    t, vd = 150, 32
    v = torch.randint(-2 ** 22 + 1, 2 ** 22, (1, t, 1, vd), generator=gen).float() / 2 ** 12
    k = torch.zeros(1, t, 1, kd)
    k[..., 5] = 1.
    args = [x.to(device) for x in (k, v, torch.zeros(1, t, 1), torch.ones(1, t, 1))]
    final = scan(None, *args, None, chunk=64, offset=0)[2]
    want = torch.zeros_like(final)
    want[:, :, 5] = v[:, -1].to(device)
    return final, want


@pytest.mark.parametrize("kd", [16, 64, 72, 128, 256])
def test_float32_state_sums_positions_in_order(kd):
    """Each write undoes the one before (D_t = v_t - v_{t-1}).  The values are
    multiples of 2^-12 below 2^10, so that each difference, and each partial sum
    of a sum in the positions' order (it is v_t), is a float32 number: the
    final state is the last value exactly.  In another order the partial sums
    need more bits."""
    from gpa_amd.ops import gdn_scan_hip
    final, want = telescoping(gdn_scan_hip, DEV, kd)
    assert torch.equal(final, want)


def exact_order(scan, device, kd=16):
    """[(got, want)] of one-token float32 scans whose sums are exact in the
    recurrences' order only.  The key has 1/2 at keys 0, 4, 5 and 8 and writes are
    full; rows of the state there are 2 A, 2 B, -2 B and 2 t with t far below an ulp of
    A and B.  D = U - W S with U = A is A - A - B + B - t; where the sum over the keys
    comes before U, or key 8 before key 5, t is lost.  dD = dd0 + Kn dS is the same
    sum.  The state's new row is e^G S + k D with the product rounded and e^G S
    added to it in one rounding."""
    gen = torch.Generator().manual_seed(6)
    vd = 32
    odd = lambda lo, hi: (2 * torch.randint(lo // 2, hi // 2, (vd,), generator=gen) + 1).float()
    a, b, t = odd(2 ** 21, 2 ** 22), odd(2 ** 21, 2 ** 22), odd(1, 2 ** 10) / 2 ** 14
    k = torch.zeros(1, 1, 1, kd)
    k[..., [0, 4, 5, 8]] = 0.5

    def rows(*x):
        s = torch.zeros(1, 1, kd, vd)
        s[0, 0, [0, 4, 5, 8]] = torch.stack(x)
        return s

    one, zero = torch.ones(1, 1, 1), torch.zeros(1, 1, 1)
    v = a.view(1, 1, 1, vd)
    move = lambda *xs: [x.to(device).requires_grad_() for x in xs]
    out = []
    args = move(k, k, v, zero, one, rows(2 * a, 2 * b, -2 * b, 2 * t))
    got = scan(*args, chunk=64, offset=0)
    out.append((got[2][0, 0, 8], 1.5 * t))
    dv, = torch.autograd.grad([got[0], got[2]], [args[2]],
                              [v.to(device), rows(-2 * a, 2 * b, -2 * b, 2 * t).to(device)])
    out.append((dv.flatten(), t))

    s0 = rows(*torch.randn(4, vd, generator=gen))
    s0[0, 0, 8] = 0.  # the new row is k D
    s0[0, 0, 1] = 1.  # ... and e^G
    v = torch.randn(1, 1, 1, vd, generator=gen)
    final = scan(None, *move(k, v, zero - 0.3, one, s0), chunk=64, offset=0)[2][0, 0].detach().double().cpu()
    out.append((final[0], (final[1] * s0[0, 0, 0].double() + final[8]).float()))
    return [(x.detach().float().cpu(), y) for x, y in out]


@pytest.mark.parametrize("kd", [16, 18, 128, 256])
def test_float32_state_sums_in_the_recurrences_order(kd):
    from gpa_amd.ops import gdn_scan_hip
    for got, want in exact_order(gdn_scan_hip, DEV, kd):
        assert torch.equal(got, want)
