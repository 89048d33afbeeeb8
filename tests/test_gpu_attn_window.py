"""Sliding-window attention (bf16, head_dim 64) where a window's edge meets a
wave's 32 queries or a 64-key tile, against float64.

The bound: each weight is rounded to bf16 (2^-9 of it, the sum taken over the
rounded ones), so the output is off by 2^-8 sum p |v| / sum p, and by its own
rounding, 2^-9 of it; fp32 sums lie far below (doubled for them)."""
import ctypes as C

import numpy as np
import pytest

import snapjudge_amd as sj

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("window", [1, 31, 32, 33, 63, 64, 65, 96, 200])
def test_window_edges(window):
    print(f"window {window}", flush=True)
    B, L, H = 3, 333, 2
    lens = [333, 129, 64]
    g = torch.Generator(device="cuda").manual_seed(window)
    qkv = torch.randn(B, L, 3, H, 64, generator=g, device="cuda").bfloat16()
    out = torch.full((B, L, H * 64), 7.0, dtype=torch.bfloat16, device="cuda")
    dl = torch.tensor(lens, dtype=torch.int32, device="cuda")
    P = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
    sj.check(sj.lib().sjh_attn(P(qkv), P(dl), P(out), B, L, H, 64, window, sj.SJH_BF16, None))
    x, got = qkv.double().cpu().numpy(), out.double().cpu().numpy().reshape(B, L, H, 64)
    i = np.arange(L)
    for b, n in enumerate(lens):
        near = np.abs(i[:, None] - i[None, :n]) <= window
        live = near.any(1)
        for h in range(H):
            assert np.all(got[b, ~live, h] == 0)
            s = np.where(near, x[b, :, 0, h] @ x[b, :n, 1, h].T / 8.0, -np.inf)[live]
            p = np.exp(s - s.max(1, keepdims=True))
            p /= p.sum(1, keepdims=True)
            want = p @ x[b, :n, 2, h]
            lim = 2 * (2.0 ** -8 * (p @ np.abs(x[b, :n, 2, h])) + 2.0 ** -9 * np.abs(want))
            assert np.all(np.abs(got[b, live, h] - want) <= lim), (b, h)
