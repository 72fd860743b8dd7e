"""What ulm_decode_step refuses before it launches anything, and which sizes it
takes. The addresses here are made up: every call returns from the checks."""
import ctypes

import pytest

import ulm_native as nat

P = ctypes.c_void_p
POINTERS = ["norm_w", "conv_w", "key_w", "key_b", "log_eps", "val_w", "mu_w", "w", "g", "conv_buf", "S", "c", "r_prev",
            "pv", "pr"]


class Layer(ctypes.Structure):
    _fields_ = [(n, P) for n in POINTERS] + [("norm_eps", ctypes.c_double), ("pending", ctypes.c_longlong)]


def _refusal(n_layers=2, **change):
    """The message of a call whose last layer has `change`."""
    layers = (Layer * n_layers)(*[Layer(*[P(1 << 20)] * 15, 1e-5, 3) for _ in range(n_layers)])
    for k, v in change.items():
        setattr(layers[n_layers - 1], k, v)
    N, D, A, Kc = 2, 64, 128, 4
    need = nat.lib().ulm_decode_step_workspace_bytes(N, D, A, Kc)
    status = nat.lib().ulm_decode_step(layers, n_layers, P(1 << 21), P(1 << 22), P(1 << 23), need, N, D, A, Kc, None)
    assert status != nat.ULM_OK
    return nat.lib().ulm_last_error().decode()


@pytest.mark.parametrize("name", ["mu_w", "w", "S", "c", "r_prev", "pr"])
def test_refuses_misaligned_pointers(name):
    """Read or written 16 bytes at a time, pr by the write-back of the 16th term."""
    assert "must be 16-byte aligned" in _refusal(**{name: (1 << 20) + 4})


@pytest.mark.parametrize("change", [{n: None} for n in POINTERS] + [{"pending": 16}, {"pending": -1}])
def test_refuses_null_pointers_and_full_states(change):
    message = _refusal(**change)
    assert "ulm_decode_step: " in message and "layer 1" in message


def test_sizes():
    """Up to 256 sequences, 4096 slots in fours, 8 taps, features whose row fits 60 KB."""
    takes = lambda *s: nat.lib().ulm_decode_step_workspace_bytes(*s) > 0  # noqa: E731
    assert takes(256, 64, 128, 4) and not takes(257, 64, 128, 4)
    assert takes(1, 64, 4096, 4) and not takes(1, 64, 4100, 4) and not takes(1, 64, 126, 4)
    assert takes(1, 64, 128, 8) and not takes(1, 64, 128, 9) and takes(1, 64, 128, 1)
    assert takes(1, 15360, 4, 4) and not takes(1, 15361, 4, 4)


@pytest.mark.parametrize("N,D,A,taken", [
    (256, 64, 128, True), (256, 64, 1024, True), (128, 288, 712, True), (16, 768, 3072, True), (32, 768, 3072, True),
    (40, 512, 3072, True), (1, 288, 712, True), (8, 768, 3072, True),
    (64, 768, 3072, False), (48, 768, 2048, False), (256, 288, 712, False), (128, 768, 768, False),
    (256, 512, 512, False), (256, 768, 128, False), (256, 64, 4096, False), (256, 32, 4096, False), (100, 1600, 400, False),
])
def test_takes_the_sizes_it_is_faster_at(N, D, A, taken):
    """Both sides of the line between this form and the per-kernel one, by what each took there."""
    assert (nat.lib().ulm_decode_step_workspace_bytes(N, D, A, 4) > 0) == taken
