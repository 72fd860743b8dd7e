"""The two-launch decode position (ulm_decode_step) against
the per-kernel form of UnifiedBlock.step, position by position through two
write-backs, and the calls it leaves to that form (needs an MI355X). Both are
fp32 evaluations of the same sums in other orders: outputs, S, c and r_prev
agree to 1e-6 of their size, 16 roundings of 6e-8."""
import pytest
import torch

from helpers import rel, say

pytestmark = pytest.mark.gpu

import model as model_mod  # noqa: E402
from model import ModelArgs, UnifiedBlock, UnifiedLM  # noqa: E402


def _block(D, A, taps, seed, n_layers=1):
    torch.manual_seed(seed)
    lm = UnifiedLM(ModelArgs(dim=D, hidden_dim=A, n_layers=n_layers, vocab_size=50, conv_size=taps,
                             norm_eps=1e-12)).eval()
    with torch.no_grad():
        for b in lm.layers:
            b.conv.weight.normal_(std=0.5)
            b.key.weight.normal_(std=D ** -0.5)
            b.key.bias.normal_(std=0.3)
            b.val.weight.normal_(std=D ** -0.5)
            b.log_rate.fill_(-3.0)
            b.log_w.normal_(std=0.5)
    return lm.cuda()


# sequences on both sides of each register width, feature counts on and off the 32-row tiles and the 64-wide and
# 768-wide column slices, groups of sequences cut by 16, by the LDS and by 4, slot counts of every slice count and cut inside a lane's last slice
CASES = [(1, 288, 712, 4), (1, 7, 4, 1), (2, 768, 3072, 4), (3, 100, 1000, 2), (4, 262, 36, 8), (5, 64, 256, 4),
         (8, 768, 3072, 4), (9, 33, 2052, 3), (16, 768, 1280, 4), (7, 1024, 4096, 4), (1, 1600, 128, 4), (17, 72, 520, 4), (45, 1024, 260, 4), (256, 40, 64, 4)]


@pytest.mark.parametrize("N,D,A,taps", CASES)
def test_matches_per_kernel_step(N, D, A, taps, monkeypatch):
    say(f"two-launch decode step N={N} D={D} A={A} taps={taps}")
    block = _block(D, A, taps, N * D + A).layers[0]
    gen = torch.Generator(device="cuda").manual_seed(3)
    new, old = (block.init_state(N, torch.device("cuda")) for _ in range(2))
    took = []
    real = model_mod.decode_step
    for t in range(35):
        # small beside what the block adds, so that the output's own rounding does not hide an error there
        x = 1e-4 * torch.randn(N, D, device="cuda", generator=gen)
        monkeypatch.setattr(model_mod, "decode_step", lambda *a: took.append(real(*a)) or took[-1])
        got = block.step(x, new)
        monkeypatch.setattr(model_mod, "decode_step", lambda *a: None)
        ref = block.step(x, old)
        # the sums' roundings (the address's, q's and the read-out's, 6e-8 each), and the outputs' own
        err = (got - ref).norm().item()
        bound = 2e-6 * (ref - x).norm().item() + 1.2e-7 * x.norm().item()
        assert err <= bound and new["np"] == old["np"], (t, err, bound)
    assert len(took) == 35 and all(o is not None for o in took)
    block.flush_state(new), block.flush_state(old)
    errs = {k: rel(new[k], old[k]) for k in ("S", "c", "r_prev", "buf") if old[k].numel()}
    say(f"  rel {errs}")
    assert max(errs.values()) < 1e-6, errs


@pytest.mark.parametrize("N", [1, 6])
def test_whole_model_takes_one_call(N, monkeypatch):
    say(f"UnifiedLM.step N={N}: every block in one call against block by block")
    lm = _block(96, 140, 4, 5, n_layers=3)
    tokens = torch.randint(0, 50, (20, N), device="cuda")
    a, b = lm.init_states(N, "cuda"), lm.init_states(N, "cuda")
    calls = []
    real = model_mod.decode_step
    monkeypatch.setattr(model_mod, "decode_step", lambda x, s, e: calls.append(len(s)) or real(x, s, e))
    got = [lm.step(t, a) for t in tokens]
    assert calls == [3] * 20
    monkeypatch.setattr(model_mod, "decode_step", lambda *a: None)
    ref = [lm.step(t, b) for t in tokens]
    assert rel(torch.stack(got), torch.stack(ref)) < 1e-6
    assert all(s["np"] == 4 for s in a)


def test_left_to_the_per_kernel_form():
    """Too many sequences, a strided state, a state and weights that disagree: nothing is touched."""
    block = _block(64, 128, 4, 1).layers[0]
    say("calls the two-launch step leaves alone")
    for N, change in ((257, None), (4, "strided"), (4, "short")):
        s = block.init_state(N, torch.device("cuda"))
        block._pending(s, torch.device("cuda"))
        if change == "strided":
            s["c"] = torch.zeros(128, N, device="cuda").t()
        if change == "short":
            s["S"] = torch.zeros(N, 64, 124, device="cuda")
        before = {k: s[k].clone() for k in ("S", "c", "r_prev", "buf")}
        assert model_mod.decode_step(torch.randn(N, 64, device="cuda"), [s], [1e-5]) is None
        assert s["np"] == 0 and all(torch.equal(s[k], t) for k, t in before.items())


def test_final_norm_in_one_launch():
    """The step's last norm against the module: rsqrt of a D-term mean, a few roundings of 6e-8; a hooked norm
    goes through its module."""
    lm = _block(100, 64, 4, 2)
    say("UnifiedLM.step: the final norm in one launch")
    with torch.no_grad():
        lm.norm.weight.normal_()
        h = torch.randn(5, 100, device="cuda")
        assert rel(lm._final_norm(h), lm.norm(h)) < 1e-6
        seen = []
        lm.norm.register_forward_hook(lambda m, i, o: seen.append(o))
        lm.step(torch.zeros(2, dtype=torch.long, device="cuda"), lm.init_states(2, "cuda"))
    assert len(seen) == 1


@pytest.mark.parametrize("form", [tuple, iter, lambda states: dict(enumerate(states)).values()])
def test_states_in_any_iterable(form):
    """UnifiedLM.step takes its states from any iterable, and no more of them than it has blocks."""
    lm = _block(96, 140, 4, 5, n_layers=3)
    say("UnifiedLM.step: states in a tuple, an iterator, a view")
    a, b = lm.init_states(2, "cuda"), lm.init_states(2, "cuda")
    for t in range(3):
        tokens = torch.tensor([t, t + 1], device="cuda")
        assert torch.equal(lm.step(tokens, form(a)), lm.step(tokens, b))
    more = iter(a + ["left"])
    lm.step(tokens, more)
    assert next(more) == "left"


class _Sub(torch.Tensor):
    pass


@pytest.mark.parametrize("where,key,change", [
    ("state", "pr", "misaligned"), ("state", "S", "misaligned"), ("state", "S", "subclass"), ("state", "c", "negative"),
    ("params", "w", "negative"), ("params", "mu_w", "subclass"), ("params", "mu_w", "misaligned")])
def test_tensors_left_to_the_per_kernel_form(where, key, change):
    """Tensors off 16 bytes, subclasses and lazily negated ones: nothing is touched."""
    say(f"the two-launch step leaves a {change} {key} of the {where} alone")
    block = _block(64, 128, 4, 1).layers[0]
    s = block.init_state(3, torch.device("cuda"))
    block._pending(s, torch.device("cuda"))
    held = s if where == "state" else s["params"]
    t = held[key]
    if change == "misaligned":
        held[key] = torch.zeros(t.numel() + 1, device="cuda")[1:].view(t.shape).copy_(t)
    else:
        held[key] = t.as_subclass(_Sub) if change == "subclass" else torch._neg_view(t)
    before = {k: s[k].detach().clone() for k in ("S", "c", "r_prev", "buf")}
    assert model_mod.decode_step(torch.randn(3, 64, device="cuda"), [s], [1e-5]) is None
    assert s["np"] == 0 and all(torch.equal(s[k], t) for k, t in before.items())
