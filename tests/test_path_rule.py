"""Which form serves a training shape on the 32 grid past the flop comparison
(train_path in csrc/fm_ops.hip, ulm_fm_path): the block-pair form where the
state form's workgroups are few, on both sides of each of the rule's lines, and
the two forms' agreement at shapes that take it."""
import pytest
import torch

import ulm_native as nat

CHUNKED, PAIR = 1, 2


@pytest.mark.parametrize("B,T,A,D,form", [
    (8, 512, 128, 64, PAIR),       # 16 workgroups: 1.3 times the state form's flops
    (2, 2048, 512, 256, PAIR),     # 16 workgroups: 1.9 times
    (4, 2048, 128, 64, PAIR),      # 8 workgroups: 5.1 times
    (64, 1024, 128, 64, PAIR),     # 128 workgroups: 2.6 times, the line at 3.2
    (128, 1024, 128, 64, CHUNKED),  # 256 workgroups: 2.6 times, the line at 1.7
    (8, 128, 64, 32, CHUNKED),     # one tile of positions
    (8, 129, 64, 32, PAIR),
    (1, 2048, 256, 128, PAIR),
    (1, 2049, 256, 128, CHUNKED),  # past 2048 positions
    (20, 2048, 128, 64, PAIR),     # 503 MB of saved scores
    (21, 2048, 128, 64, CHUNKED),  # 528 MB
])
def test_rule(B, T, A, D, form, monkeypatch):
    monkeypatch.delenv("ULM_FM_PATH", raising=False)
    assert nat.lib().ulm_fm_path(B, T, A, D) == form


@pytest.mark.gpu
@pytest.mark.parametrize("B,T,A,D", [(8, 512, 128, 64), (2, 129, 64, 32), (1, 2048, 256, 128)])
def test_forms_agree(B, T, A, D, monkeypatch):
    """Outputs and gradients of the rule's form and the state form, both bf16 products with fp32 sums: each is
    within 1e-2 of float64 in the parity cases, so within 2e-2 of the other."""
    import workloads
    from helpers import rel, say
    from kernel import unified_memory
    say(f"block-pair and state form B={B} T={T} A={A} D={D}")
    r, v, g, w = workloads.block_inputs(B, T, D, A, seed=T, device=torch.device("cuda"), v_dtype=torch.bfloat16)
    res = []
    for form in ("", "chunked"):
        monkeypatch.setenv("ULM_FM_PATH", form)
        leaves = [t.detach().clone().requires_grad_(True) for t in (r, v, g, w)]
        q, fast = unified_memory(*leaves)
        grads = torch.autograd.grad((q, fast), leaves, (0.1 * q.detach(), fast.detach()))
        res.append([q, fast, *grads])
    errs = [rel(a, b) for a, b in zip(*res)]
    say(f"  {errs}")
    assert max(errs) < 2e-2, errs
