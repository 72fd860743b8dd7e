"""The forward statistics (fwd_stats_kernel) at the edges of its chunks, groups
of chunks, slot blocks and segments, through unified_memory's q, which it forms
in fp32 (needs an MI355X). q = r / c with c a decayed sum of at most T
non-negative terms: 16-term fp32 sums joined by powers of lam, so a relative
error of some ten roundings of 6e-8 against float64."""
import pytest
import torch

from helpers import say

pytestmark = pytest.mark.gpu

import ulm_native as nat  # noqa: E402
from kernel import unified_memory  # noqa: E402
from ulm_native import call, ptr  # noqa: E402


def _q64(r, lam, w):
    n = torch.zeros_like(r[:, 0])
    q = torch.empty_like(r)
    for t in range(r.shape[1]):
        n = lam * n + (r[:, t - 1] if t else 0)
        q[:, t] = r[:, t] / (w + n)
    return q


@pytest.mark.parametrize("B,T,A", [(1, 1, 1), (2, 16, 63), (1, 17, 64), (3, 64, 65), (1, 65, 130), (2, 127, 200),
                                   (1, 193, 96), (1, 1024, 70), (1, 1025, 33), (2, 2113, 40), (260, 65, 30)])
def test_q_against_float64(B, T, A):
    say(f"forward statistics B={B} T={T} A={A}")
    gen = torch.Generator().manual_seed(T * A)
    r = (torch.randn(B, T, A, generator=gen).clamp(min=0) ** 2 / A).cuda()
    w = (4 * torch.exp(torch.randn(A, generator=gen))).cuda()
    v = torch.randn(B, T, 8, generator=gen).cuda()
    g = torch.tensor(-0.02, device="cuda")
    q, _ = unified_memory(r, v, g, w)
    ref = _q64(r.double(), torch.exp(g.double()), w.double())
    assert ((q.double() - ref).abs() <= 1e-6 * ref.abs()).all()


@pytest.mark.parametrize("T", [65, 200, 1030])
def test_rows_do_not_depend_on_the_batch(T):
    """A few rows take two chunks side by side, many one: the same bits."""
    say(f"forward statistics of one row alone and among 300, T={T}")
    gen = torch.Generator().manual_seed(T)
    r = torch.rand(300, T, 70, generator=gen).cuda() / 70
    v = torch.randn(300, T, 8, generator=gen).cuda()
    g, w = torch.tensor(-0.1, device="cuda"), torch.full((70,), 2.0, device="cuda")
    q, fast = unified_memory(r, v, g, w)
    for b in (0, 151, 299):
        q1, f1 = unified_memory(r[b:b + 1].contiguous(), v[b:b + 1].contiguous(), g, w)
        assert torch.equal(q1[0], q[b]) and torch.equal(f1[0], fast[b])


def test_prior_masses_at_the_ends_of_the_range():
    """A mass whose reciprocal overflows, huge, infinite and zero ones: r / c as a division gives it."""
    say("forward statistics: denormal, huge, infinite and zero prior masses")
    T, w = 70, torch.tensor([1e-39, 1e-37, 3e38, float("inf"), 0.0, 1.0], device="cuda")
    r = torch.zeros(1, T, 6, device="cuda")
    r[0, T - 1] = 0.25   # no evidence before it: c = w
    v = torch.ones(1, T, 4, device="cuda")
    q, _ = unified_memory(r, v, torch.tensor(-0.5, device="cuda"), w)
    got, want = q[0, T - 1].cpu(), (r[0, T - 1] / w).cpu()
    assert torch.equal(got, want), (got, want)
    assert torch.equal(q[0, :T - 1, :4], torch.zeros(T - 1, 4, device="cuda"))


# ---- the address formed from pre (the fused block's input kind), w q out, the prefill's c and decayed keys

def _block_rows(pre, bias, denom, v, g, w, x, prefill):
    """(w q, x + fast[, S, c]) of ulm_block_fm_fwd or ulm_block_fm_prefill."""
    (B, T, A), D = pre.shape, v.shape[-1]
    dt, lib = nat.dtype_code(pre.dtype), nat.lib()
    qw, y = torch.empty_like(pre), torch.empty(B, T, D, device="cuda")
    outs = [qw, y]
    head = (ptr(pre), dt, ptr(bias), ptr(denom), ptr(v), dt, ptr(g), ptr(w), ptr(qw), dt, ptr(x), ptr(y))
    if prefill:
        S, c = torch.empty(B, D, A, device="cuda"), torch.empty(B, A, device="cuda")
        wb = lib.ulm_block_fm_prefill_workspace_bytes(B, T, A, D, dt)
        ws = torch.empty(wb, device="cuda", dtype=torch.uint8)
        call("ulm_block_fm_prefill", *head, ptr(S), ptr(c), ptr(ws), wb, B, T, A, D, nat.stream_of(pre))
        outs += [S, c]
    else:
        sb, wb = lib.ulm_fm_saved_bytes(B, T, A, D, dt), lib.ulm_block_fm_fwd_workspace_bytes(B, T, A, D)
        saved, ws = (torch.empty(n, device="cuda", dtype=torch.uint8) for n in (sb, wb))
        call("ulm_block_fm_fwd", *head, ptr(saved), sb, ptr(ws), wb, B, T, A, D, nat.stream_of(pre))
    return outs


@pytest.mark.parametrize("prefill", [False, True])
@pytest.mark.parametrize("path", ["pair", "chunked", "generic"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T", [1, 65, 200, 1030])
def test_formed_address_alone_and_among_many(T, dtype, path, prefill, monkeypatch):
    """One row (two chunks side by side) and among 140 of two slot blocks each (one): the same bits of w q, the
    output and the decode state, and w q and c against float64. c: some ten fp32 roundings, and lam = exp(g) an ulp
    off, 1.2e-7, over a mean lag of 1 / 0.03 positions; w q the same or its dtype's rounding (2^-8, 2^-11)."""
    monkeypatch.setenv("ULM_FM_PATH", path)
    B, A, D = 140, 96, 32
    say(f"formed address of one row alone and among {B}, T={T} {dtype} {path} prefill={prefill}")
    gen = torch.Generator(device="cuda").manual_seed(T)
    rn = lambda *s: torch.randn(*s, device="cuda", generator=gen)  # noqa: E731
    pre, v, x, bias = rn(B, T, A).to(dtype), rn(B, T, D).to(dtype), rn(B, T, D), 0.2 * rn(A)
    g, w, le, denom = torch.full((1,), -0.03, device="cuda"), torch.exp(rn(A)), torch.zeros(1, device="cuda"), rn(B, T)
    call("ulm_addr_fwd", ptr(pre), nat.dtype_code(dtype), ptr(bias), ptr(le), None, ptr(denom), B * T, A, nat.stream_of(pre))
    many = _block_rows(pre, bias, denom, v, g, w, x, prefill)
    for b in (0, B - 1):
        cut = lambda t: t[b:b + 1].contiguous()  # noqa: E731
        alone = _block_rows(cut(pre), bias, cut(denom), cut(v), g, w, cut(x), prefill)
        for i, (one, all_) in enumerate(zip(alone, many)):
            assert torch.equal(one[0], all_[b]), (b, i)
    z = (pre.double() + bias.double()).clamp(min=0).square()
    r, lam = z / (1 + z.sum(-1, keepdim=True)), torch.exp(g.double())
    want = _q64(r, lam, w.double()) * w.double()
    tol = 1e-6 + 1.2e-7 / 0.03
    rel = {torch.float32: tol, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    # fp16 keeps 2^-24 of absolute precision below 2^-14
    assert ((many[0].double() - want).abs() <= rel * want.abs() * 1.01 + (2.0 ** -24 if dtype == torch.float16 else 0)).all()
    if prefill:
        n = torch.zeros_like(r[:, 0])
        for t in range(T):
            n = lam * n + (r[:, t - 1] if t else 0)
        assert ((many[3].double() - (w.double() + n)).abs() <= tol * (w.double() + n)).all()


@pytest.mark.parametrize("w", [3e38, 9e37, 5e37, 1.5e36, 1e36, 1e-36, 8e-37, 7e-37, 2e-38, 1e-38, 1e-39])
def test_quotients_of_huge_and_tiny_masses(w):
    """A wave of one such mass: r / c as a division gives it, quotients below 2^-126 and reciprocals there included."""
    say(f"forward statistics: every prior mass {w}")
    T, A = 70, 64
    gen = torch.Generator(device="cuda").manual_seed(1)
    r = torch.zeros(1, T, A, device="cuda")
    r[0, T - 1] = torch.rand(A, device="cuda", generator=gen) * 2.0 ** torch.randint(-20, 1, (A,), device="cuda", generator=gen)
    w = torch.full((A,), w, device="cuda")
    q, _ = unified_memory(r, torch.ones(1, T, 4, device="cuda"), torch.tensor(-0.5, device="cuda"), w)
    want = (r[0, T - 1].double() / w.double()).float()
    got, fin = q[0, T - 1], torch.isfinite(want)
    assert torch.equal(torch.isinf(got), ~fin)   # overflows as a division's
    # an ulp of the quotient (2^-149 below 2^-126)
    assert ((got[fin].double() - want[fin].double()).abs() <= want[fin].double() * 2.0 ** -23 + 2.0 ** -149).all()


def test_keys_whose_sum_nears_the_largest_float():
    """A key of 1e38 makes the masses after it huge and their quotients denormal; the reads through the same key are of
    ordinary size and want those quotients."""
    say("forward statistics: a huge key")
    T, A = 40, 32
    r = torch.rand(1, T, A, device="cuda") / A
    r[0, 3] = 1e38
    q, _ = unified_memory(r, torch.ones(1, T, 4, device="cuda"), torch.tensor(-0.01, device="cuda"), torch.ones(A, device="cuda"))
    ref = _q64(r.double(), torch.exp(torch.tensor(-0.01, device="cuda").double()), torch.ones(A, device="cuda").double())
    assert ((q.double() - ref).abs() <= 2e-6 * ref + 2.0 ** -149).all()
