"""Attention with fp32 products at the edges of its tiles, against float64.

The bound: a score is a sum of Dh products, off by ds = (Dh + 3) 2^-24 scale
max_j sum |q k_j|; a weight relative to the largest is then off by 2 ds + 8
2^-24 (its score, the maximum's, expf) and a sum of n weights or weighted values
by n 2^-24 more; the quotient of two such sums by twice that, times max |v|.
bf16 outputs add one rounding."""
import ctypes as C

import numpy as np
import pytest

import snapjudge_amd as sj

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


# rows and keys at the edges of a wave's 16 queries, a workgroup's 64 and a key
# tile's 64 (32 at head_dim 128); no keys; a window narrower than a tile and one
# that spans two; head dims padded to a block (8), of one to eight blocks
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("Dh", [8, 16, 32, 64, 128])
@pytest.mark.parametrize("L,window", [(1, 0), (17, 0), (64, 3), (65, 0), (130, 0), (200, 70)])
def test_attn_f32_edges(Dh, L, window, dtype):
    if dtype == "bf16" and Dh == 64:
        pytest.skip("the bf16 head_dim-64 kernel")
    print(f"attn f32 Dh={Dh} L={L} window={window} {dtype}", flush=True)
    H = 2
    lens = sorted({0, 1, L // 2, max(L - 1, 0), L})
    B = len(lens)
    g = torch.Generator(device="cuda").manual_seed(L + Dh)
    qkv = torch.randn(B, L, 3, H, Dh, generator=g, device="cuda")
    qkv = qkv.bfloat16() if dtype == "bf16" else qkv
    out = torch.full((B, L, H * Dh), 7.0, dtype=qkv.dtype, device="cuda")
    dl = torch.tensor(lens, dtype=torch.int32, device="cuda")
    P = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
    sj.check(sj.lib().sjh_attn(P(qkv), P(dl), P(out), B, L, H, Dh, window, sj.SJH_BF16 if dtype == "bf16" else sj.SJH_F32, None))
    x, got = qkv.double().cpu().numpy(), out.double().cpu().numpy().reshape(B, L, H, Dh)
    u, scale = 2.0 ** -24, Dh ** -0.5
    far = np.abs(np.arange(L)[:, None] - np.arange(L)[None]) > window if window else np.zeros((L, L), bool)
    for b, n in enumerate(lens):
        for h in range(H):
            q, k, v = x[b, :, 0, h], x[b, :n, 1, h], x[b, :n, 2, h]
            dead = far[:, :n].all(1) if n else np.ones(L, bool)
            assert np.all(got[b, dead, h] == 0)  # no key to read
            if n == 0:
                continue
            s = np.where(far[:, :n], -np.inf, q @ k.T * scale)[~dead]
            p = np.exp(s - s.max(1, keepdims=True))
            want = (p / p.sum(1, keepdims=True)) @ v
            ds = (Dh + 3) * u * scale * (np.abs(q) @ np.abs(k).T).max(1)[~dead]
            lim = (2 * (2 * ds + (n + 8) * u) * np.abs(v).max())[:, None] + (2.0 ** -8 * np.abs(want) if dtype == "bf16" else 0)
            assert np.all(np.abs(got[b, ~dead, h] - want) <= lim), (b, h)


@pytest.mark.parametrize("key", [72, 90, 135, 150, 170, 199])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_attn_f32_infinite_rows_past_the_window(key, bad):
    # an infinite or NaN V row reaches the queries of a 64-query block that has it
    # in some query's window, and no others: their values are as without it
    print(f"attn f32 V row {key} {bad}", flush=True)
    L, H, Dh, window = 200, 2, 64, 8
    g = torch.Generator(device="cuda").manual_seed(key)
    qkv = torch.randn(1, L, 3, H, Dh, generator=g, device="cuda")
    dl = torch.tensor([L], dtype=torch.int32, device="cuda")
    P = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
    outs = []
    for v in (None, bad):
        if v is not None:
            qkv[0, key, 2] = v
        out = torch.full((L, H * Dh), 7.0, device="cuda")
        sj.check(sj.lib().sjh_attn(P(qkv), P(dl), P(out), 1, L, H, Dh, window, sj.SJH_F32, None))
        outs.append(out.cpu())
    block = torch.arange(L) // 64 * 64
    free = (key < block - window) | (key >= block + 64 + window)
    seen = (torch.arange(L) - key).abs() <= window
    assert torch.equal(outs[1][free], outs[0][free])
    assert not torch.isfinite(outs[1][seen]).any()
