"""The row sums of the norm + conv kernels, bit for bit (needs an MI355X). A row's
sum over channels is, in each 64-channel wave, the halving tree over lanes 32,
16, .. 1 apart whose first step adds the lower lane's product unrounded to the
upper lane's rounded one, and then the waves' sums in order: the oracle here
does that in float32 on the CPU (a product of two floats is exact in float64,
and one rounding of the sum to float32 follows)."""
import numpy as np
import pytest
import torch

from helpers import say

pytestmark = pytest.mark.gpu

import ulm_native as nat  # noqa: E402
from ulm_native import call, ptr  # noqa: E402

F = np.float32


def _fma(a, b, c):
    return (a.astype(np.float64) * b.astype(np.float64) + c.astype(np.float64)).astype(F)


def _row_sums(a, b):
    """Sum over the last dimension of a * b, float32, in the kernels' order."""
    D = a.shape[-1]
    pad = [(0, 0)] * (a.ndim - 1) + [(0, -D % 64)]
    a, b = (np.pad(t, pad).reshape(*t.shape[:-1], -1, 64) for t in (a, b))
    v = _fma(a[..., :32], b[..., :32], a[..., 32:] * b[..., 32:])
    while v.shape[-1] > 1:
        half = v.shape[-1] // 2
        v = v[..., :half] + v[..., half:]
    total = np.zeros(v.shape[:-2], F)
    for w in range(v.shape[-2]):
        total = total + v[..., w, 0]
    return total


def _fwd(x, nw, cw, h, u, rstd):
    (B, T, D), Kc = x.shape, cw.shape[1]
    # eps = 0: the mean square is one rounding of the sum over D
    call("ulm_norm_conv_fwd", ptr(x), nat.ULM_F32, ptr(nw), ptr(cw), Kc, 0.0, ptr(h), nat.ULM_F32, ptr(u), nat.ULM_F32,
         ptr(rstd), B, T, D, nat.stream_of(x))


def _rsqrt(mean):
    """The kernel's own rsqrt of the means: rows of two channels whose squares' float32 sum is twice the mean."""
    two = 2 * mean
    x0 = np.sqrt(two)
    while (x0 * x0 > two).any():
        x0 = np.where(x0 * x0 > two, np.nextafter(x0, F(0)), x0)
    x1 = np.sqrt(two - x0 * x0)
    assert (x0 * x0 + x1 * x1 == two).all()
    x = torch.from_numpy(np.stack([x0, x1], -1).reshape(1, -1, 2)).cuda()
    one, rstd = torch.ones(2, device="cuda"), torch.empty(x.shape[:2], device="cuda")
    _fwd(x, one, one[:, None].contiguous(), torch.empty_like(x), torch.empty_like(x), rstd)
    return rstd.view(mean.shape)


@pytest.mark.parametrize("B,T,D,Kc", [(2, 16, 64, 4), (1, 1, 7, 1), (3, 37, 100, 8), (2, 50, 768, 4), (1, 33, 1024, 3)])
def test_rstd_and_dx(B, T, D, Kc):
    say(f"norm + conv row sums B={B} T={T} D={D} Kc={Kc}")
    gen = torch.Generator().manual_seed(T * D + Kc)
    rn = lambda *s: torch.randn(*s, generator=gen)  # noqa: E731
    x, nw, cw, du = rn(B, T, D), 1 + 0.1 * rn(D), rn(D, Kc), rn(B, T, D)
    xd, nwd, cwd, dud = (t.cuda() for t in (x, nw, cw, du))
    h, u, dx = (torch.empty(B, T, D, device="cuda") for _ in range(3))
    rstd, dnw, dcw = torch.empty(B, T, device="cuda"), torch.empty(D, device="cuda"), torch.empty(D, Kc, device="cuda")
    _fwd(xd, nwd, cwd, h, u, rstd)
    xn = x.numpy()
    mean = _row_sums(xn, xn) * (F(1) / F(D))
    assert torch.equal(rstd, _rsqrt(mean))

    wsb = nat.lib().ulm_norm_conv_bwd_workspace_bytes(B, T, D, Kc)
    ws = torch.empty(wsb, device="cuda", dtype=torch.uint8)
    call("ulm_norm_conv_bwd", ptr(xd), nat.ULM_F32, ptr(rstd), ptr(nwd), ptr(cwd), Kc, ptr(dud), nat.ULM_F32, None,
         nat.ULM_F32, None, ptr(dx), ptr(dnw), ptr(dcw), ptr(ws), wsb, B, T, D, nat.stream_of(xd))
    r, n, c, g = rstd.cpu().numpy()[..., None], nw.numpy(), cw.numpy(), du.numpy()
    g = np.pad(g, [(0, 0), (0, Kc - 1), (0, 0)])
    dh = np.zeros_like(xn)
    for m in range(Kc):   # dh_t = sum_m cw[Kc - 1 - m] du_{t+m}
        dh = _fma(np.broadcast_to(c[:, Kc - 1 - m], dh.shape), g[:, m:m + T], dh)
    xn, an = xn * r, dh * n
    dot = _row_sums(xn, an) * (F(1) / F(D))
    want = r * _fma(-xn, np.broadcast_to(dot[..., None], xn.shape), an)
    assert torch.equal(dx.cpu(), torch.from_numpy(want))
