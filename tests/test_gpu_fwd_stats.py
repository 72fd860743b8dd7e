"""The forward statistics (fwd_stats_kernel) at the edges of its chunks, groups
of chunks, slot blocks and segments, through unified_memory's q, which it forms
in fp32 (needs an MI355X). q = r / c with c a decayed sum of at most T
non-negative terms: 16-term fp32 sums joined by powers of lam, so a relative
error of some ten roundings of 6e-8 against float64."""
import pytest
import torch

from helpers import say

pytestmark = pytest.mark.gpu

from kernel import unified_memory  # noqa: E402


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
