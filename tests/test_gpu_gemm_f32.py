"""The fp32-product GEMM at the edges of its tiles, against float64.

The bound is the standard one for a dot product of K terms in fp32, whatever
the order of the sum: |error| <= (K + 2) 2^-24 sum |a_k w_k| (the + 2 for the
bias or residual add and the store)."""
import ctypes as C

import numpy as np
import pytest

import snapjudge_amd as sj

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def P(t):
    return C.c_void_p(t.data_ptr()) if t is not None else None


def bound(a, w, K, extra):
    return (K + 2) * 2.0 ** -24 * (np.abs(a) @ np.abs(w).T + np.abs(extra))


# 64x64 tiles (enough of them for every CU), 16x64 and 16x16 tiles whose waves
# split K; row and column remainders; K of one step, a partial last step
# (772, 30), fewer steps than waves (48), rows no vector load can read (51)
@pytest.mark.parametrize("M,N,K", [(1090, 1027, 96), (1025, 1024, 772), (300, 1500, 772), (257, 1024, 51), (16, 768, 768),
                                   (1, 256, 772), (33, 17, 48), (7, 1, 768), (15, 2, 256), (5, 300, 51), (3, 70, 4),
                                   (130, 64, 30)])
def test_gemm_f32_edges(M, N, K):
    print(f"gemm f32 M={M} N={N} K={K}", flush=True)
    rng = np.random.default_rng(M + 7 * N + K)
    a, w, b, x = (rng.standard_normal(s).astype(np.float32) for s in ((M, K), (N, K), (N,), (M, N)))
    A, W, B, X = (torch.from_numpy(v).cuda() for v in (a, w, b, x))
    out = torch.full((M + 1, N), 7.0, device="cuda")
    a, w = a.astype(np.float64), w.astype(np.float64)
    prod = a @ w.T
    sj.check(sj.lib().sjh_gemm(P(A), P(W), P(B), P(out), M, N, K, 0, sj.SJH_F32, None))
    got = out.cpu().numpy()
    assert np.all(np.abs(got[:M] - (prod + b)) <= bound(a, w, K, b[None] + 0 * prod))
    assert np.all(got[M] == 7.0)  # nothing past the last row
    sj.check(sj.lib().sjh_gemm_residual(P(A), P(W), P(X), M, N, K, sj.SJH_F32, None))
    assert np.all(np.abs(X.cpu().numpy() - (prod + x)) <= bound(a, w, K, x))


@pytest.mark.parametrize("M,F,K", [(17, 33, 64), (600, 1152, 96), (1100, 512, 64)])
def test_gemm_f32_geglu_pairs(M, F, K):
    # the input and gate halves of a tile meet in the epilogue, at partial last
    # column tiles too; the GELU's slope is at most 1.13 and |gelu(u)| <= |u|
    print(f"geglu f32 M={M} F={F} K={K}", flush=True)
    rng = np.random.default_rng(M + F)
    a, w = (rng.standard_normal(s).astype(np.float32) for s in ((M, K), (2 * F, K)))
    out = torch.empty((M, F), device="cuda")
    A, W = torch.from_numpy(a).cuda(), torch.from_numpy(w).cuda()
    sj.check(sj.lib().sjh_gemm_geglu(P(A), P(W), P(out), M, F, K, sj.SJH_F32, None))
    a, w = a.astype(np.float64), w.astype(np.float64)
    u = a @ w.T
    act = 0.5 * u[:, :F] * (1 + torch.erf(torch.from_numpy(u[:, :F] / np.sqrt(2.0))).numpy())
    e = bound(a, w, K, 0 * u)
    lim = 1.13 * e[:, :F] * np.abs(u[:, F:]) + np.abs(u[:, :F]) * e[:, F:] + e[:, :F] * e[:, F:]
    lim += 8 * 2.0 ** -24 * (np.abs(u[:, :F]) + 1) * (np.abs(u[:, F:]) + 1)  # erff, its argument, the products
    assert np.all(np.abs(out.cpu().numpy() - act * u[:, F:]) <= lim)


# 32- and 64-row tiles staged through registers: rows no vector load can read,
# steps ending inside a piece of four values, K of less than a step, bf16 rows
# (products exact in fp32; a bf16 store rounds by at most 2^-8 of its value)
@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("M,N,K", [(300, 1500, 51), (257, 1601, 772), (2100, 2050, 16), (2049, 2111, 3), (2100, 2050, 70)])
def test_gemm_f32_staged_through_registers(M, N, K, dtype):
    print(f"gemm staged {dtype} M={M} N={N} K={K}", flush=True)
    rng = np.random.default_rng(M + 5 * N + K)
    td, code = (torch.bfloat16, sj.SJH_BF16) if dtype == "bf16" else (torch.float32, sj.SJH_F32)
    A, W = (torch.from_numpy(rng.standard_normal(s).astype(np.float32)).to(td) for s in ((M, K), (N, K)))
    a, w, b = A.double().numpy(), W.double().numpy(), rng.standard_normal(N).astype(np.float32)
    A, W, B = A.cuda(), W.cuda(), torch.from_numpy(b).cuda()
    out = torch.full((M + 1, N), 7.0, device="cuda", dtype=td)
    sj.check(sj.lib().sjh_gemm(P(A), P(W), P(B), P(out), M, N, K, 0, code, None))
    got, ref = out.cpu().double().numpy(), a @ w.T + b
    lim = bound(a, w, K, b[None] + 0 * ref) + (2.0 ** -8 * np.abs(ref) if dtype == "bf16" else 0)
    lim *= 1 + 2.0 ** -8  # the store rounds the computed value, not the exact one
    assert np.all(np.abs(got[:M] - ref) <= lim)
    assert np.all(got[M] == 7.0)


def test_gemm_f32_more_tiles_than_one_grid_dimension_holds():
    # 2^24 tiles of 256 threads: gelu(x) * y of one product each, so that every
    # value is known; the output is 33 GB
    M, F = 65, 1 << 28
    if torch.cuda.mem_get_info()[0] < 60 << 30:
        pytest.skip("needs 60 GB of free device memory")
    print(f"geglu M={M} F={F} K=1", flush=True)
    A = torch.ones(M, 1, dtype=torch.bfloat16, device="cuda")
    A[-1] = 2
    W = torch.ones(2 * F, 1, dtype=torch.bfloat16, device="cuda")
    out = torch.zeros(M, F, dtype=torch.bfloat16, device="cuda")
    sj.check(sj.lib().sjh_gemm_geglu(P(A), P(W), P(out), M, F, 1, sj.SJH_BF16, None))
    for r in (0, 1, 31, 32, 63, 64):
        x = 2.0 if r == M - 1 else 1.0
        want = x * 0.5 * x * (1 + float(torch.erf(torch.tensor(x / 2 ** 0.5, dtype=torch.float64))))
        lo, hi = float(out[r].min()), float(out[r].max())
        assert lo == hi and abs(lo - want) <= 2.0 ** -8 * want, r
