"""The host module's eager calls (csrc/host.cpp) against the registered ops and
the Python implementations they stand in for, bit for bit, and the calls that
it leaves to those (needs an MI355X)."""
import pytest
import torch

from helpers import say

pytestmark = pytest.mark.gpu

import kernel  # noqa: E402
import ulm_native as nat  # noqa: E402
from model import ModelArgs, UnifiedBlock  # noqa: E402


def _args(B, T, D, A, taps, seed, form="plain", bias=True):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rn = lambda *s, std=1.0: torch.randn(*s, device="cuda", generator=gen) * std  # noqa: E731
    x = rn(B, T, D)
    key = rn(A, D, std=D ** -0.5)
    if form == "strided":   # an input and a weight that are views in another order
        x, key = rn(T, B, D).transpose(0, 1), rn(D, A, std=D ** -0.5).t()
    if form == "half":      # weights kept in bf16
        key = key.to(torch.bfloat16)
    t = [x, 1 + rn(D, std=0.1), rn(D, 1, taps, std=0.5), key, rn(A, std=0.1) if bias else None,
         torch.zeros((), device="cuda"), rn(D, D, std=D ** -0.5), rn(D, A, std=0.05), torch.tensor(-3.0, device="cuda"),
         rn(A, std=0.4)]
    return [None if a is None else a.detach().requires_grad_(True) for a in t], rn(B, T, D)


BLOCKS = [(2, 70, 64, 96, 4, "plain", True), (1, 1, 7, 5, 1, "plain", True), (3, 130, 40, 70, 8, "strided", True),
          (2, 33, 96, 128, 3, "plain", False), (2, 200, 288, 712, 4, "half", True)]


@pytest.mark.parametrize("cdt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,T,D,A,taps,form,bias", BLOCKS)
def test_block_equals_registered_op(B, T, D, A, taps, form, bias, cdt):
    say(f"host block vs registered op B={B} T={T} D={D} A={A} taps={taps} {form} {cdt}")
    args, dout = _args(B, T, D, A, taps, T + D, form, bias)
    leaves = [a for a in args if a is not None]
    got = kernel.block_eager(*args, 1e-5, cdt)
    assert got is not None
    g1 = torch.autograd.grad(got, leaves, dout)
    ref = kernel.block_fwd(*args, 1e-5, cdt)[0]
    g2 = torch.autograd.grad(ref, leaves, dout)
    for a, b in zip((got, *g1), (ref, *g2)):
        assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b)


@pytest.mark.parametrize("cdt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,T,D,A,taps,form,bias", BLOCKS)
def test_prefill_equals_python(B, T, D, A, taps, form, bias, cdt):
    say(f"host prefill vs block_prefill B={B} T={T} D={D} A={A} taps={taps} {form} {cdt}")
    args, _ = _args(B, T, D, A, taps, T + D, form, bias)
    out, S, c, r_prev, buf, g, w = kernel.block_prefill_eager(*args, 1e-5, cdt)
    ref = kernel.block_prefill(*args, 1e-5, cdt)
    for a, b in zip((out, S, c, r_prev), ref):
        assert torch.equal(a, b)
    n = min(taps - 1, T)
    want = torch.zeros(B, D, taps - 1, device="cuda")
    if n:
        want[:, :, taps - 1 - n:] = ref[4][:, T - n:].float().transpose(1, 2)
    assert torch.equal(buf, want) and not out.requires_grad
    assert torch.equal(g[0], -torch.exp(args[8])) and torch.equal(w, torch.exp(args[9].clamp(-7, 12)))


@pytest.mark.parametrize("which", ["both", "q", "fast"])
def test_memory_equals_registered_op(which):
    say(f"host unified_memory vs registered op, gradients of {which}")
    gen = torch.Generator(device="cuda").manual_seed(2)
    r = torch.rand(2, 90, 70, device="cuda", generator=gen).to(torch.bfloat16) / 70
    v = torch.randn(90, 2, 40, device="cuda", generator=gen).transpose(0, 1).to(torch.bfloat16)
    g, w = torch.tensor(-0.05, device="cuda"), torch.full((70,), 4.0, device="cuda")
    res = []
    for host in (True, False):
        leaves = [t.detach().clone().requires_grad_(True) for t in (r, v, g, w)]
        out = nat.host().memory(*leaves) if host else kernel.fm_fwd(*leaves)[:2]
        outs = {"both": out, "q": out[:1], "fast": out[1:]}[which]
        grads = torch.autograd.grad(outs, leaves, [torch.ones_like(o) for o in outs])
        res.append([*out, *grads])
    for a, b in zip(*res):
        assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b)


def test_left_to_the_registered_ops():
    say("calls the host module leaves alone")
    args, _ = _args(2, 40, 32, 64, 4, 1)
    host = nat.host()
    take = lambda a, cdt=torch.float32: host.block(1e-5, cdt, *a)  # noqa: E731
    assert take(args) is not None
    swap = lambda i, t: args[:i] + [t] + args[i + 1:]  # noqa: E731
    assert take(args, torch.float64) is None
    assert take(swap(0, args[0].double())) is None and take(swap(0, args[0][0])) is None
    assert take(swap(3, args[3].cpu())) is None and take(swap(9, args[9][:-1])) is None

    class Sub(torch.Tensor):
        pass
    assert take(swap(0, args[0].detach().as_subclass(Sub))) is None
    seen = []

    def loss(x):
        seen.append(take(swap(0, x)))
        return kernel.block_fwd(x, *args[1:], 1e-5, torch.float32)[0].square().sum()
    with pytest.raises(RuntimeError, match="functorch"):   # refused by the registered op, as without the host module
        torch.func.grad(loss)(args[0].detach())
    assert seen == [None]
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(args[0].detach(), torch.ones_like(args[0]))
        assert take(swap(0, dual)) is None


def test_saved_tensor_hooks_see_what_is_saved():
    """Offloading hooks pack and unpack every tensor a block saves, inputs and intermediates."""
    say("saved-tensor hooks over a block")
    args, dout = _args(2, 40, 32, 64, 4, 1)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t.cpu(), lambda t: t.cuda()):
        out = kernel.block_eager(*args, 1e-5, torch.float32)
    assert len(packed) == 19
    got = torch.autograd.grad(out, args, dout)
    ref = torch.autograd.grad(kernel.block_eager(*args, 1e-5, torch.float32), args, dout)
    assert all(torch.equal(a, b) for a, b in zip(got, ref))


def test_module_forward_under_autocast():
    say("UnifiedBlock.forward: the autocast dtype reaches the host path")
    torch.manual_seed(0)
    block = UnifiedBlock(ModelArgs(dim=64, hidden_dim=96)).cuda()
    x = torch.randn(2, 50, 64, device="cuda")
    with torch.autocast("cuda", dtype=torch.bfloat16):
        got = block(x)
    p = block
    ref = kernel.block_fwd(x, p.norm.weight, p.conv.weight, p.key.weight, p.key.bias, p.log_eps, p.val.weight,
                           p.mu.weight, p.log_rate, p.log_w, p.norm.eps, torch.bfloat16)[0]
    assert torch.equal(got, ref) and got.requires_grad


def _block_leaves(bias=True):
    args, dout = _args(2, 40, 32, 64, 4, 1, bias=bias)
    return args, [a for a in args if a is not None], dout


def _memory_leaves(parameter):
    gen = torch.Generator(device="cuda").manual_seed(4)
    r = (torch.rand(2, 40, 96, device="cuda", generator=gen) / 96).requires_grad_(True)
    v = torch.randn(2, 40, 64, device="cuda", generator=gen).requires_grad_(True)
    g, w = torch.tensor(-0.05, device="cuda", requires_grad=True), torch.full((96,), 4.0, device="cuda")
    return [r, v, g, torch.nn.Parameter(w) if parameter else w.requires_grad_(True)]


@pytest.mark.parametrize("which", ["block", "block without bias", "memory", "memory with a Parameter"])
def test_second_derivative_raises(which):
    """create_graph gives the first gradients, the same bits, and a second backward is refused: no term of it may
    vanish without an error."""
    say(f"second derivatives of {which}")
    if which.startswith("block"):
        args, leaves, _ = _block_leaves("without" not in which)
        call = lambda: kernel.unified_block(*args, 1e-5).square().sum()  # noqa: E731
    else:
        leaves = _memory_leaves("Parameter" in which)
        call = lambda: sum(t.square().sum() for t in kernel.unified_memory(*leaves))  # noqa: E731
    first = torch.autograd.grad(call(), leaves)
    loss = call()
    again = torch.autograd.grad(loss, leaves, create_graph=True)
    assert all(a.requires_grad and torch.equal(a, b) for a, b in zip(again, first))
    with pytest.raises(RuntimeError, match="no autograd formula"):
        (loss + again[0].square().sum()).backward()


@pytest.mark.parametrize("which", ["block", "block without bias", "memory", "memory, q alone"])
def test_batch_of_gradients(which):
    """is_grads_batched: the vmapped backward, against one backward for each gradient."""
    say(f"a batch of gradients through {which}")
    if which.startswith("block"):
        args, leaves, dout = _block_leaves("without" not in which)
        out = kernel.unified_block(*args, 1e-5)
    else:
        leaves = _memory_leaves(True)
        out = kernel.unified_memory(*leaves)[0 if "alone" in which else 1]
        leaves = leaves if "alone" not in which else [leaves[0], leaves[2], leaves[3]]
    gen = torch.Generator(device="cuda").manual_seed(9)
    ups = torch.randn(3, *out.shape, device="cuda", generator=gen)
    got = torch.autograd.grad(out, leaves, ups, is_grads_batched=True, retain_graph=True)
    each = [torch.autograd.grad(out, leaves, u, retain_graph=True) for u in ups]
    for a, b in zip(got, zip(*each)):
        assert torch.equal(a, torch.stack(b))


def test_gradient_with_a_negative_bit():
    """A gradient that is a lazily negated view counts with its sign."""
    say("a gradient with the negative bit")
    args, leaves, dout = _block_leaves()
    out = kernel.unified_block(*args, 1e-5)
    got = torch.autograd.grad(out, leaves, torch._neg_view(dout), retain_graph=True)
    ref = torch.autograd.grad(out, leaves, -dout)
    assert all(torch.equal(a, b) for a, b in zip(got, ref))


@pytest.mark.parametrize("which", ["memory", "block", "prefill", "copies", "decode_step"])
def test_other_threads_run_during_a_call(which):
    """The interpreter's lock is free while a call works: with no forced switch for 1000 s, a thread that waits for
    the lock gets it inside one of the calls or never."""
    import sys
    import threading
    import time
    say(f"another thread runs during {which}")
    host = nat.host()
    args, _ = _args(2, 300, 96, 128, 4, 3)
    args = [a.detach() for a in args]
    if which == "memory":
        leaves = [t.detach() for t in _memory_leaves(False)]
        call = lambda: host.memory(*leaves)  # noqa: E731
    elif which == "copies":
        call = lambda: host.copies(args[3], args[7], args[6])  # noqa: E731
    elif which == "decode_step":
        block = UnifiedBlock(ModelArgs(dim=64, hidden_dim=128)).cuda()
        s = block.init_state(2, torch.device("cuda"))
        block._pending(s, torch.device("cuda"))
        x = torch.randn(2, 64, device="cuda")
        call = lambda: host.decode_step(x, [s], [1e-5])  # noqa: E731
    else:
        call = lambda: getattr(host, which)(1e-5, torch.float32, *args)  # noqa: E731
    assert call() is not None
    torch.cuda.synchronize()
    ran, kept, gate = [], [], threading.Lock()
    gate.acquire()

    def other():
        with gate:
            ran.append(True)
    thread = threading.Thread(target=other)
    thread.start()
    time.sleep(0.1)   # it waits at the gate
    before = sys.getswitchinterval()
    sys.setswitchinterval(1000)
    try:
        gate.release()
        for _ in range(2000):
            kept.append(call())   # dropping a tensor frees the lock for a moment by itself
            if ran:
                break
        seen = bool(ran)
    finally:
        sys.setswitchinterval(before)
    thread.join()
    assert seen


def test_function_modes_see_the_registered_op():
    """A torch function mode sees the block's op, as without the host module; a default device is none."""
    from torch.overrides import TorchFunctionMode
    say("a block under a torch function mode and under a default device")
    args, _ = _args(2, 40, 32, 64, 4, 1)
    seen = []

    class Mode(TorchFunctionMode):
        def __torch_function__(self, func, types, a=(), kw=None):
            seen.append(str(func))
            return func(*a, **(kw or {}))
    ref = kernel.block_eager(*args, 1e-5, torch.float32)
    with Mode():
        assert kernel.block_eager(*args, 1e-5, torch.float32) is None
        got = kernel.unified_block(*args, 1e-5)
    assert "ulm.block_fwd.default" in seen and torch.equal(got, ref)
    with torch.device("cuda"):
        assert kernel.block_eager(*args, 1e-5, torch.float32) is not None


def _all_calls(dout, args, leaves, block):
    """One pass through every eager entry: memory and block with their backwards, a prefill, then decode steps."""
    q, fast = kernel.unified_memory(*leaves)
    out = [q, fast, *torch.autograd.grad((q, fast), leaves, (0.1 * q.detach(), fast.detach()))]
    y = kernel.unified_block(*args, 1e-5)
    out += [y, *torch.autograd.grad(y, args, dout)]
    y, s = block.prefill(args[0].detach())
    out += [y]
    for t in range(18):
        out.append(block.step(y[:, t], s))
    block.flush_state(s)
    return [t.clone() for t in out + [s["S"], s["c"], s["r_prev"], s["buf"]]]


def _problem(seed):
    args, dout = _args(2, 150, 64, 128, 4, seed)
    torch.manual_seed(seed)
    return dout, args, _memory_leaves(False), UnifiedBlock(ModelArgs(dim=64, hidden_dim=128)).cuda()


def test_on_another_stream():
    """Every eager entry on a stream of the caller's, the inputs' writes and the outputs' reads on it too: the
    same bits as on the default stream."""
    say("the eager calls on another stream")
    ref = _all_calls(*_problem(5))
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    for _ in range(3):
        with torch.cuda.stream(stream):
            torch.cuda._sleep(20_000_000)   # a launch on any other stream would run ahead of the inputs
            got = _all_calls(*_problem(5))
        stream.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, ref))


def test_from_two_threads():
    """Two threads, each with its stream, state and inputs, at once: each gets its own results."""
    import threading
    say("the eager calls from two threads at once")
    refs = [_all_calls(*_problem(s)) for s in (5, 6)]
    torch.cuda.synchronize()
    problems = [_problem(s) for s in (5, 6)]
    torch.cuda.synchronize()
    got, start = [None, None], threading.Barrier(2)

    def work(i):
        stream = torch.cuda.Stream()
        start.wait()
        with torch.cuda.stream(stream):
            got[i] = [_all_calls(*problems[i]) for _ in range(5)]
        stream.synchronize()
    threads = [threading.Thread(target=work, args=(i,)) for i in (0, 1)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i in (0, 1):
        assert got[i] is not None
        for one in got[i]:
            assert all(torch.equal(a, b) for a, b in zip(one, refs[i]))
