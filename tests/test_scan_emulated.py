"""The chunked GDN scan's kernels (gdn_scan.hip and the prep, 256-key state,
out / dd0, late-read and chunk-backward MFMA kernels) built for the host and run under
AddressSanitizer (tests/host_emu/), against the oracle's per-token
recurrence in float64 (reference ops.py:29-85), on the CPU.

The cases reach the float32 FMA path (state, out and dd0 kernels of
gdn_scan.hip, the chunk backward on fp32 MFMA, or the FMA chunk backward
when K is not a multiple of 4), the bfloat16 FMA path (K not a multiple of
16) and the bfloat16 MFMA path in each key-width class (64, 128 and 256, with
K below and at the tile; widths, and rows off 16-byte boundaries, that take the
element-wise loads of the preparation and leave the fragment chunk backward),
with chunk offsets, ragged last chunks and tiny shapes.  Every global access of
those kernels is checked against the exact extent of the buffer it addresses
(each of a scan's intermediates, fragments and scratch buffers in a tensor of
its own), and new memory is NaN; the results are held to the GPU tests' bar:
relative L2 1e-4 in float32, 2e-2 in bfloat16.  The strip state kernels that
bfloat16 scans of at most 128 keys take are not emulated (their LDS loads are
inline global_load_lds): a plain recurrence stands in for them
(host_emu/strip_reference.cpp), and the GPU tests cover them.
"""
import ctypes
import ctypes.util

import pytest
import torch

from tests.host_emu import harness
from tests.test_gpu_gdn_scan import _inputs, _oracle_segments, _oracle_segments_autograd, _rel
from tests.test_gpu_gdn_state_f32 import exact_order, telescoping

CASES = [
    # (B, T, H, K, V, chunk, offset, dtype)
    (2, 9, 2, 4, 3, 4, 2, torch.float32),
    (2, 11, 1, 6, 5, 4, 1, torch.float32),  # K % 4 != 0: the FMA chunk backward at 64 keys
    (1, 40, 2, 40, 24, 16, 5, torch.bfloat16),  # K % 16 != 0: the bfloat16 FMA state path
    (1, 70, 2, 32, 48, 64, 17, torch.float32),
    (1, 40, 1, 256, 64, 16, 3, torch.float32),
    (1, 40, 1, 256, 64, 64, 3, torch.float32),
    (1, 40, 1, 128, 64, 16, 3, torch.float32),
    (1, 129, 1, 256, 96, 64, 1, torch.bfloat16),
    (1, 70, 1, 192, 128, 64, 5, torch.bfloat16),
    (1, 9, 1, 16, 8, 8, 3, torch.bfloat16),
    (1, 70, 1, 48, 20, 64, 5, torch.bfloat16),  # V % 8 != 0: element-wise rows, the general chunk backward
    (1, 70, 2, 64, 40, 64, 17, torch.bfloat16),
    (1, 40, 1, 80, 96, 16, 3, torch.bfloat16),
    (1, 129, 1, 128, 64, 64, 1, torch.bfloat16),
]
IDS = [f"B{c[0]}T{c[1]}H{c[2]}K{c[3]}V{c[4]}C{c[5]}o{c[6]}{str(c[7])[6:]}" for c in CASES]


@pytest.fixture
def host(host_runner, monkeypatch, tmp_path):
    from gpa_amd import ops
    harness.use_host(monkeypatch, harness.HostLib(host_runner, str(tmp_path)))
    monkeypatch.setattr(ops, "_pieces", harness.SeparateBuffers())
    # host tensors belong to no stream: nothing to mark as in use
    monkeypatch.setattr(ops, "_in_use_here", lambda *tensors: None)
    was = torch.are_deterministic_algorithms_enabled(), torch.is_deterministic_algorithms_warn_only_enabled()
    torch.use_deterministic_algorithms(True, warn_only=True)  # new tensors start as NaN
    yield
    torch.use_deterministic_algorithms(was[0], warn_only=was[1])


def test_every_scan_buffer_is_an_allocation_of_its_size(host, monkeypatch):
    """What the host run bounds: each intermediate and each scratch buffer ends
    where its allocation does."""
    from gpa_amd.ops import gdn_scan_hip
    seen, locate = set(), harness.HostLib._locate

    def check(self, spans, p):
        i, at = locate(self, spans, p)
        seen.add(spans[i][1])
        assert at == 0, "a buffer inside another's allocation"
        return i, at

    monkeypatch.setattr(harness.HostLib, "_locate", check)
    q, k, v, g, beta, s0 = (x.requires_grad_() for x in _inputs(1, 9, 1, 16, 8, torch.bfloat16, seed=1))
    out, _, final = gdn_scan_hip(q, k, v, g, beta, s0, chunk=64, offset=0)
    (out.float().sum() + final.sum()).backward()
    # one chunk of one stream: float32 kn, delta, u (a whole strip) and T, bf16 w and k fragments
    assert {64 * 16 * 4, 64 * 8 * 4, 64 * 32 * 4, 64 * 64 * 4, 2 * 64 * 16 * 2, 4 * 64 * 16 * 2} <= seen


@pytest.mark.parametrize("case", CASES, ids=IDS)
def test_emulated_scan_forward_matches_recurrence(host, case):
    from gpa_amd.ops import gdn_scan_hip
    b, t, h, kd, vd, chunk, offset, dtype = case
    q, k, v, g, beta, s0 = _inputs(b, t, h, kd, vd, dtype, seed=11)
    out, states, final = gdn_scan_hip(q, k, v, g, beta, s0, chunk=chunk, offset=offset)
    ref_out, ref_states, ref_final = _oracle_segments(q, k, v, g, beta, s0, chunk, offset)
    tol = 1e-4 if dtype == torch.float32 else 2e-2
    errs = dict(out=_rel(out, ref_out), states=_rel(states, ref_states), final=_rel(final, ref_final))
    print(case, errs)
    assert all(e < tol for e in errs.values()), errs


@pytest.mark.parametrize("case", CASES, ids=IDS)
@pytest.mark.parametrize("with_q", [True, False], ids=["read", "noread"])
def test_emulated_scan_backward_matches_autograd_of_recurrence(host, case, with_q):
    """Gradients of a loss over the read, the chunk-start states (injected
    into the backward) and the final state.  The float32 cases above 128
    keys run the FMA chunk backward (gdn_chunk_bwd<float, 256>), whose dA
    product once read rows of an LDS matrix that other threads were already
    overwriting: a race the host build's independent threads expose."""
    from gpa_amd.ops import gdn_scan_hip
    b, t, h, kd, vd, chunk, offset, dtype = case
    q, k, v, g, beta, s0 = _inputs(b, t, h, kd, vd, dtype, seed=5, q=with_q)
    gen = torch.Generator().manual_seed(3)
    nch = (offset + t + chunk - 1) // chunk
    w_out = torch.randn(b, t, h, vd, generator=gen, dtype=torch.float64)
    w_states = torch.randn(b, h, nch, kd, vd, generator=gen, dtype=torch.float64) * .1
    w_final = torch.randn(b, h, kd, vd, generator=gen, dtype=torch.float64)

    def loss(out, states, final):
        total = (final.double() * w_final).sum() + (states.double() * w_states).sum()
        return total + (out.double() * w_out).sum() if out is not None else total

    leaves = [x.clone().requires_grad_() if x is not None else None for x in (q, k, v, g, beta, s0)]
    out, states, final = gdn_scan_hip(*leaves, chunk=chunk, offset=offset)
    loss(out if with_q else None, states, final).backward()
    refs = [x.detach().double().requires_grad_() if x is not None else None for x in (q, k, v, g, beta, s0)]
    ro, rs, rf = _oracle_segments_autograd(refs[:3], refs[3], refs[4], refs[5], chunk, offset)
    loss(ro if with_q else None, rs, rf).backward()
    tol = 1e-4 if dtype == torch.float32 else 2e-2
    names = ["dq", "dk", "dv", "dg", "dbeta", "ds0"]
    errs = {n: _rel(a.grad, r.grad) for n, a, r in zip(names, leaves, refs) if a is not None}
    print(case, with_q, errs)
    assert all(e < tol for e in errs.values()), errs


def test_emulated_float32_state_sums_positions_in_order(host):
    """Keys that all point one way and full writes: every position's write undoes
    the one before (D_t = v_t - v_{t-1}).  The values are multiples of 2^-12 below 2^10,
    so that each difference, and each partial sum of a sum in the positions'
    order (it is v_t), is a float32 number: the final state is the last value
    exactly.  In any other order the partial sums need more bits."""
    from gpa_amd.ops import gdn_scan_hip
    final, want = telescoping(gdn_scan_hip, "cpu")
    assert torch.equal(final, want)


@pytest.mark.parametrize("kd", [16, 18, 128])
def test_emulated_float32_state_sums_in_the_recurrences_order(host, kd):
    from gpa_amd.ops import gdn_scan_hip
    for got, want in exact_order(gdn_scan_hip, "cpu", kd):
        assert torch.equal(got, want)


@pytest.mark.parametrize("dtype,kd", [(torch.float32, 16), (torch.float32, 100), (torch.bfloat16, 16)], ids=str)
def test_emulated_inverse_of_parallel_keys(host, monkeypatch, dtype, kd):
    """T = (I + A)^-1 for keys that all point one way, where A_ts = beta_t exactly
    and the terms of T's sums cancel from row to row: summed in order, no partial
    sum is above a few times T's elements (of at most 1) and its error stays below
    two roundings, 2^-23 of its norm (the host build rounds the products of the
    diagonal blocks too); where four rows apart are added first it is larger."""
    from gpa_amd import ops
    k = torch.zeros(1, 64, 1, kd, dtype=dtype)
    k[..., 3] = 2.
    beta = (torch.randn(1, 64, 1, generator=torch.Generator().manual_seed(2)) + 2).sigmoid()
    ops.gdn_scan_hip(None, k, torch.ones(1, 64, 1, 8, dtype=dtype), torch.zeros(1, 64, 1), beta, None, chunk=64)
    work = next(b for _, b in ops._pieces.made.values() if b[2 if dtype == torch.float32 else 3] is not None and len(b) == 8)
    tri = work[5].view(64, 64).double()
    a = beta.double().view(64, 1).expand(64, 64).tril(-1)
    err = _rel(tri, torch.linalg.inv(torch.eye(64, dtype=torch.float64) + a))
    print(err)
    assert err < 2 ** -23


def _chain_order(n):
    """Contraction indices in the order in which mma8 adds them."""
    return [8 * g + s + 4 * h for g in range(n // 8) for s in range(4) for h in range(2)]


@pytest.mark.parametrize("kd,vd", [(16, 8), (80, 20)])
def test_emulated_bf16_preparation_rounds_like_the_float32_products(host, kd, vd):
    """The bf16 chunk preparation's float32 intermediates, bit for bit: the row
    norms are sums over keys 64, 32, 16, .. 1 apart, W = T diag(b e^G) Kn and U =
    T diag(b) V chains of fused multiply-adds in mma8's order over the float32
    scaled operands, W leaving as bf16 hi and lo.  (An equal result in another
    order flips bf16 roundings of everything that follows.)"""
    from gpa_amd import ops
    fmaf = ctypes.CDLL(ctypes.util.find_library("m")).fmaf
    fmaf.restype, fmaf.argtypes = ctypes.c_float, [ctypes.c_float] * 3
    _, k, v, _, beta, _ = _inputs(1, 64, 1, kd, vd, torch.bfloat16, seed=3)
    ops.gdn_scan_hip(None, k, v, torch.zeros(1, 64, 1), beta, None, chunk=64)
    work = next(b for _, b in ops._pieces.made.values() if len(b) == 8)
    frag = next(b for _, b in ops._pieces.made.values() if len(b) == 5)
    u, tri, bet = work[3], work[5].view(64, 64), work[7]
    k16, rb = kd // 16, -(-kd // 32)

    keys = torch.nn.functional.pad(k[0, :, 0].float(), (0, -kd % 64)).unflatten(1, (-1, 64))
    tree = torch.zeros(64, 64)
    for i in range(keys.shape[1]):
        tree = (tree.double() + keys[:, i].double().square()).float()  # (one rounding: a fused multiply-add)
    for apart in (32, 16, 8, 4, 2, 1):
        tree = tree + tree[:, torch.arange(64) ^ apart]
    kn = (k[0, :, 0].float() / tree[:, :1].sqrt().clamp_min(1e-6)).bfloat16()
    # krow piece (t/32, k/16), lane t%32 + 32 ((k/8) % 2), element k%8
    krow = frag[2].view(2, k16, 2, 32, 8).permute(0, 3, 1, 2, 4).reshape(64, kd)
    assert torch.equal(krow, kn)

    def product(scale, right):  # T diag(scale) right
        left, out = (tri * scale).tolist(), torch.zeros(64, right.shape[1])
        cols = right.t().tolist()
        for t in range(64):
            for j, col in enumerate(cols):
                acc = 0.
                for c in _chain_order(64):
                    acc = fmaf(left[t][c], col[c], acc)
                out[t, j] = acc
        return out

    w = product(bet, kn.float())
    hi = w.bfloat16()
    lo = (w - hi.float()).bfloat16()
    wrow = frag[0].view(2, k16, 2, 2, 32, 8).permute(2, 0, 4, 1, 3, 5).reshape(2, 64, kd)
    assert torch.equal(wrow, torch.stack((hi, lo)))
    # wcol piece (k/32, t/16), lane k%32 + 32 ((t/8) % 2), element t%8
    wcol = frag[1].view(rb, 4, 2, 2, 32, 8).permute(2, 1, 3, 5, 0, 4).reshape(2, 64, 32 * rb)
    assert torch.equal(wcol[..., :kd], torch.stack((hi, lo))) and not wcol[..., kd:].any()
    # U block [v/32][t/32][(t/8) % 4][v%32 + 32 ((t/4) % 2)][t%4]
    uv = u.view(-1, 2, 4, 2, 32, 4).permute(1, 2, 3, 5, 0, 4).reshape(64, -1)
    assert torch.equal(uv[:, :vd], product(torch.ones(64), bet[:, None] * v[0, :, 0].float()))


def _off_boundary(x):
    """The same values in rows that start 2 bytes past a 16-byte boundary."""
    wide = torch.zeros(*x.shape[:-1], x.shape[-1] + 9, dtype=x.dtype)
    wide[..., 1:x.shape[-1] + 1] = x
    return wide[..., 1:x.shape[-1] + 1]


@pytest.mark.parametrize("kd,vd", [(64, 24), (128, 64)])
def test_emulated_rows_off_boundaries_give_the_same(host, kd, vd):
    """Element-wise loads of the preparation against its 16-byte loads."""
    from gpa_amd.ops import gdn_scan_hip
    q, k, v, g, beta, s0 = _inputs(1, 70, 1, kd, vd, torch.bfloat16, seed=9)
    want = gdn_scan_hip(q, k, v, g, beta, s0, chunk=64, offset=5)
    got = gdn_scan_hip(*(_off_boundary(x) for x in (q, k, v)), g, beta, s0, chunk=64, offset=5)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("kd,vd", [(48, 24), (128, 40), (144, 32)])
def test_emulated_late_read_matches_the_scan_with_its_read(host, kd, vd):
    """A read taken after its scan (gpa_gdn_read, gpa_gdn_read_backward, and the
    scan backward that takes the read's gradient): keys that end inside a 32-key
    tile leave padding in the query fragments that the chunk backward multiplies."""
    from gpa_amd.ops import gdn_scan_deferred, gdn_scan_hip
    inputs = _inputs(1, 21, 1, kd, vd, torch.bfloat16, seed=5)
    gen = torch.Generator()
    res = []
    for late in (False, True):
        leaves = [x.clone().requires_grad_() for x in inputs]
        q, rest = leaves[0], leaves[1:]
        if late:
            states, final, read = gdn_scan_deferred(*rest, chunk=64, offset=3)
            out = read(q)
        else:
            out, states, final = gdn_scan_hip(q, *rest, chunk=64, offset=3)
        w = [torch.randn(x.shape, generator=gen.manual_seed(3)).to(x.dtype) for x in (out, states, final)]
        res.append((out, *torch.autograd.grad((out, states, final), leaves, w)))
    errs = [_rel(a, b) for a, b in zip(res[1], res[0])]
    print(kd, errs)
    assert all(e < 2e-2 for e in errs), errs  # (a NaN fails)
