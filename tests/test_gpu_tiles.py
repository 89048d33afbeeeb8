"""The tile shapes that the row count chooses between: every shape, at partial
last tiles, gives a row the same bits (each product sums K in order)."""
import ctypes as C

import numpy as np
import pytest

import snapjudge_amd as sj
from snapjudge_amd import synth

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def P(t):
    return C.c_void_p(t.data_ptr()) if t is not None else None


# rows of a 1024-column product on 256 CUs: 64x64 tiles up to 1024, 128x64 up to
# 2048, 128x128 one per CU up to 4096, two per CU; the persistent kernel from 9985
# (K 192) or as soon as two 128x128 tiles per CU are full, from 8193 (K 1088)
MS = [9985, 1, 70, 1024, 1025, 2048, 2111, 4033, 4161, 8192, 8193, 9900]


@pytest.mark.parametrize("K", [192, 1088])
@pytest.mark.parametrize("kind", ["store", "geglu", "resid", "rope", "fp8"])
def test_tile_shapes_give_the_same_bits(kind, K):
    print(f"tiles {kind} K={K}", flush=True)
    N, H = 1024, 16
    g = torch.Generator(device="cuda").manual_seed(7)
    A = torch.randn(MS[0], K, generator=g, device="cuda").bfloat16()
    nw = {"geglu": 2 * N, "rope": 3 * N}.get(kind, N)
    W = (torch.randn(nw, K, generator=g, device="cuda") * 0.1).bfloat16()
    b = torch.randn(nw, generator=g, device="cuda")
    X = torch.randn(MS[0], N, generator=g, device="cuda")
    pos = (torch.arange(MS[0], dtype=torch.int32, device="cuda") * 7) % 500
    ct, st = torch.randn(500, 32, generator=g, device="cuda"), torch.randn(500, 32, generator=g, device="cuda")
    q, sc = sj.quantize_fp8(W.float().cpu().numpy())
    Q, S = torch.from_numpy(q).cuda(), torch.from_numpy(sc).cuda()
    L = sj.lib()
    first = None
    for M in MS:
        if kind == "resid":
            out = X.clone()
            rc = L.sjh_gemm_residual(P(A), P(W), P(out), M, N, K, sj.SJH_BF16, None)
            assert torch.equal(out[M:], X[M:])
        else:
            out = torch.full((MS[0], nw if kind == "rope" else N), 7.0, dtype=torch.bfloat16, device="cuda")
            if kind == "store":
                rc = L.sjh_gemm(P(A), P(W), P(b), P(out), M, N, K, 1, sj.SJH_BF16, None)
            elif kind == "geglu":
                rc = L.sjh_gemm_geglu(P(A), P(W), P(out), M, N, K, sj.SJH_BF16, None)
            elif kind == "fp8":
                rc = L.sjh_gemm_fp8w(P(A), P(Q), P(S), P(b), P(out), M, N, K, 2, None)
            else:
                rc = L.sjh_gemm_qkv_rope(P(A), P(W), P(out), P(pos), P(ct), P(st), 500, M, H, 64, K, sj.SJH_BF16, None)
            assert bool((out[M:] == 7.0).all())  # nothing past the last row
        sj.check(rc)
        first = out if first is None else first
        assert torch.equal(out[:M], first[:M]), (kind, M)
    if kind == "fp8":  # the oracle of the fp8 tiles: float64 on the decoded weights
        w = torch.from_numpy(sj.fp8_e4m3_table()[q] * sc[:, None]).double().cuda()
        want = torch.relu(A.double() @ w.t() + b.double())
        # one bf16 rounding, and the fp32 sum's (K + 2) 2^-24 of its terms
        lim = 2.0 ** -8 * want.abs() + (K + 2) * 2.0 ** -24 * (A.double().abs() @ w.abs().t() + b.double().abs())
        assert bool(((first.double() - want).abs() <= lim).all())


def test_residual_layer_norm_epilogue_at_its_smallest_launch():
    # 44 panels of three tiles (132 of 256 CUs): the residual epilogue finishes
    # the LayerNorm from 128 tiles on, with the bits of the standalone launches
    rl, enc, w = synth.make_model(**dict(synth.PRESETS["cfg2"], num_hidden_layers=2, vocab_size=2000), seed=26)
    cfg = synth.flat_cfg(rl, enc)
    ids, mask, lens = synth.make_batch(26, 480, 400, 460, 2000, seed=28)
    T = int(lens.sum())
    assert 43 * 256 < T <= 12 * 1024
    print(f"residual LayerNorm T={T}", flush=True)
    h = []
    for fuse in (1, 0, 2):
        m = sj.Model(w, cfg, precision=sj.SJH_PREC_BF16, fuse_ln=fuse)
        h.append(m.encode(ids, mask))
        m.close()
    assert np.array_equal(h[0], h[1]) and np.array_equal(h[0], h[2])
