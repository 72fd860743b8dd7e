"""The scores and dscores of few 128 x 128 tiles, one wave per 32 x 32 tile
(pair_small_kernel), against the tiles that a larger batch takes (needs an
MI355X): both add the same products in the same order, so every output and
gradient of a row is the same bit for bit, but for the decay gradient and dw,
which sum over rows. At ragged lengths and widths around the 32-wide tiles, and
a contraction past one set of 8 steps in flight."""
import pytest
import torch

from helpers import rel, say

pytestmark = pytest.mark.gpu

from kernel import fm_prefill, unified_memory  # noqa: E402


@pytest.mark.parametrize("T,A,D,dtype", [(1, 32, 32, "bf16"), (31, 40, 33, "fp32"), (33, 300, 64, "bf16"),
                                         (100, 71, 288, "bf16"), (128, 128, 96, "bf16"), (130, 96, 40, "fp32"),
                                         (300, 64, 32, "bf16"), (129, 64, 96, "fp16")])
def test_rows_alone_and_among_many(T, A, D, dtype, monkeypatch):
    monkeypatch.setenv("ULM_FM_PATH", "pair")
    tiles = (T + 127) // 128
    tiles = tiles * (tiles + 1) // 2
    B = 64 // tiles + 1     # one row more than the few-tiles kernel takes
    say(f"few score tiles: rows alone and among {B}, T={T} A={A} D={D} {dtype}")
    gen = torch.Generator(device="cuda").manual_seed(T + A)
    rn = lambda *s: torch.randn(*s, device="cuda", generator=gen)  # noqa: E731
    dt = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}[dtype]
    r = rn(B, T, A).clamp(min=0) ** 2 / A
    v, df, dq = rn(B, T, D).to(dt), rn(B, T, D).to(dt), 0.1 * rn(B, T, A)
    g, w = torch.tensor(-0.03, device="cuda"), 4 * torch.exp(0.3 * rn(A))

    def step(rows):
        leaves = [t.detach().clone().requires_grad_(True) for t in (r[rows], v[rows], g, w)]
        q, fast = unified_memory(*leaves)
        return [q, fast, *torch.autograd.grad((q, fast), leaves, (dq[rows], df[rows]))]

    many = step(slice(0, B))
    parts = [step(slice(b, b + 1)) for b in range(B)]
    for b in (0, B // 2, B - 1):
        for i in range(4):
            assert torch.equal(parts[b][i][0], many[i][b]), (b, i)
    for i in (4, 5):
        assert rel(sum(p[i].double() for p in parts), many[i]) < 1e-5


@pytest.mark.parametrize("T", [17, 129])
def test_prefill_rows_alone_and_among_many(T, monkeypatch):
    """The prefill's scores (no transpose, no residual) the same way."""
    monkeypatch.setenv("ULM_FM_PATH", "pair")
    B = 65
    say(f"few score tiles: prefill rows alone and among {B}, T={T}")
    gen = torch.Generator(device="cuda").manual_seed(T)
    r = torch.rand(B, T, 96, device="cuda", generator=gen) / 96
    v = torch.randn(B, T, 64, device="cuda", generator=gen).to(torch.bfloat16)
    g, w = torch.tensor(-0.03, device="cuda"), torch.full((96,), 3.0, device="cuda")
    many = fm_prefill(r, v, g, w)
    for b in (0, 64):
        for a, m in zip(fm_prefill(r[b:b + 1].contiguous(), v[b:b + 1].contiguous(), g, w), many):
            assert torch.equal(a[0], m[b])
