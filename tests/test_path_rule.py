"""Which form serves a training shape (train_path in csrc/fm_ops.hip,
ulm_fm_path): it follows the length and the widths alone, never the batch, so a
row's bits do not depend on its company, and the block-pair form (whose scores
are bf16, one rounding per pair, where the state form carries hi + lo operands
and an fp32 state) serves only shapes at which it needs fewer flops."""
import pytest
import torch

import ulm_native as nat

CHUNKED, PAIR = 1, 2


@pytest.mark.parametrize("T,A,D,form", [
    (512, 128, 64, CHUNKED),     # 1.3 times the state form's flops
    (129, 64, 32, CHUNKED), (1024, 128, 64, CHUNKED), (2048, 512, 256, CHUNKED), (2049, 256, 128, CHUNKED),
    (200, 128, 64, CHUNKED),     # 0.84 times
    (128, 128, 64, PAIR),        # 0.42 times
    (256, 1152, 288, PAIR), (1024, 2048, 512, PAIR), (1024, 3072, 768, PAIR),
    (3072, 3072, 768, CHUNKED), (8192, 3072, 768, CHUNKED),
    (999, 1912, 768, PAIR), (256, 712, 288, PAIR),   # off the 32 grid
])
def test_form_follows_length_and_widths_not_the_batch(T, A, D, form, monkeypatch):
    monkeypatch.delenv("ULM_FM_PATH", raising=False)
    assert [nat.lib().ulm_fm_path(B, T, A, D) for B in (1, 2, 8, 20, 64, 128, 512)] == [form] * 7


@pytest.mark.gpu
@pytest.mark.parametrize("B,T,A,D", [(128, 1024, 128, 64), (40, 200, 128, 64)])
def test_row_alone_and_among_many(B, T, A, D, monkeypatch):
    """A narrow shape's row in a batch that fills the device and by itself: the same bits."""
    from helpers import say
    from kernel import unified_memory
    monkeypatch.delenv("ULM_FM_PATH", raising=False)
    say(f"one row alone and among {B}, T={T} A={A} D={D}")
    gen = torch.Generator(device="cuda").manual_seed(T)
    rn = lambda *s: torch.randn(*s, device="cuda", generator=gen)  # noqa: E731
    r, v = rn(B, T, A).clamp(min=0) ** 2 / A, rn(B, T, D).to(torch.bfloat16)
    dq, df = 0.1 * rn(B, T, A), rn(B, T, D).to(torch.bfloat16)
    g, w = torch.tensor(-0.05, device="cuda"), 4 * torch.exp(0.3 * rn(A))

    def step(rows):
        leaves = [t[rows].detach().clone().requires_grad_(True) for t in (r, v)]
        out = unified_memory(*leaves, g, w)
        return [*out, *torch.autograd.grad(out, leaves, (dq[rows], df[rows]))]

    many, alone = step(slice(0, B)), step(slice(B - 1, B))
    for i, (a, m) in enumerate(zip(alone, many)):
        assert torch.equal(a[0], m[B - 1]), i
