"""A decode session's key, value and mu matrices are those of its beginning: an
in-place update of the module's weights does not reach a running one, as it does
not reach the prior mass and the decay it took along."""
import pytest
import torch

from model import ModelArgs, UnifiedBlock

NAMES = {"key_w": "key", "val_w": "val", "mu_w": "mu"}


@pytest.mark.parametrize("D,A", [(64, 128), (7, 5)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_matrices_are_copies(D, A, dtype):
    torch.manual_seed(0)
    block = UnifiedBlock(ModelArgs(dim=D, hidden_dim=A)).to(dtype)
    params = block._step_params(torch.device("cpu"))
    for key, name in NAMES.items():
        before = getattr(block, name).weight.detach().float().clone()
        with torch.no_grad():
            getattr(block, name).weight.add_(1.0)
        assert params[key].dtype == torch.float32 and params[key].is_contiguous()
        assert torch.equal(params[key], before)


@pytest.mark.gpu
@pytest.mark.parametrize("start", ["init_state", "prefill"])
@pytest.mark.parametrize("D,A", [(64, 128), (64, 130)])
def test_session_goes_on_with_its_matrices(start, D, A):
    from helpers import say
    say(f"weights updated in a running decode, {start} D={D} A={A}")
    torch.manual_seed(0)
    block = UnifiedBlock(ModelArgs(dim=D, hidden_dim=A)).cuda()
    x = torch.randn(3, 5, D, device="cuda")
    new = lambda: block.prefill(x)[1] if start == "prefill" else block.init_state(3, torch.device("cuda"))  # noqa: E731
    a, b = new(), new()
    for t in range(5):
        if t == 2:
            with torch.no_grad():
                saved = [getattr(block, n).weight.clone() for n in NAMES.values()]
                for n in NAMES.values():
                    getattr(block, n).weight.mul_(1.5)
        got = block.step(x[:, t], a)
        if t >= 2:
            with torch.no_grad():
                for n, w in zip(NAMES.values(), saved):
                    getattr(block, n).weight.copy_(w)
        assert torch.equal(got, block.step(x[:, t], b))
