"""The work that stands for this framework in use, one case per call.

A user has a DecisionModel (or its encoder) staged on the GPU once and sends it
batches: a single request with its question, a handful of short requests, a bulk
of documents to embed, a few long documents, many typed questions over shared
documents.  Programs that bring their own layers call the kernel-level entry
points on device tensors.  The widths are the two encoders the benchmark runs
(768 and 1024 hidden, heads of 64); the stacks below are those encoders cut to a
few layers, so that each case answers for its layers alone.

Every case is a dict of plain values; ``kind`` selects the entry point:
  encode   Model.encode_device on token ids in HBM -> hidden states [T, D]
  forward  Model.forward on host arrays -> logits, act probabilities, and the
           logits of the unmasked markers alone
  shared   Model.forward_shared on host arrays -> the same
  gemm     sjh_gemm on device tensors -> C [M, N]
  attn     sjh_attn on device tensors -> O [B, L, H * 64]

Row lengths follow from the case (evenly spread over [lo, hi]), their order and
every value from the seed.  The model of a case is staged once per process, as a
serving program keeps it.
"""
from __future__ import annotations

import ctypes
import functools
import math

import numpy as np
import torch

import snapjudge_amd as sj

WIDTHS = {
    "base": dict(hidden_size=768, num_attention_heads=12, intermediate_size=1152),
    "large": dict(hidden_size=1024, num_attention_heads=16, intermediate_size=2624),
}
VOCAB, MAX_POS, THETA, LOCAL, EPS, N_ACT, HEADS = 50368, 8192, 160000.0, 128, 1e-5, 2, 2
PREC = {"fp32": sj.SJH_PREC_FP32, "bf16": sj.SJH_PREC_BF16, "fp8": sj.SJH_PREC_FP8W}
# markers of a question by type: choice 4..16, score 5, yes/no 2
MARKERS = {0: (4, 16), 1: (5, 5), 2: (2, 2)}
K_MAX = 16


def listed():
    return [
        # one request as a router sends it: a short text and its question, host
        # arrays in, logits out, through the full 22-layer model (batch 1 latency)
        dict(name="request", kind="forward", width="base", prec="bf16", layers=22, local=False, B=1, lo=73, hi=73),
        # a request of a few words, encoder only: launches and latency are all there is
        dict(name="encode_tiny", kind="encode", width="base", prec="bf16", layers=4, local=False, B=1, lo=17, hi=17),
        # one full-length short request, the latency shape of the benchmark
        dict(name="encode_one", kind="encode", width="base", prec="bf16", layers=4, local=False, B=1, lo=128, hi=128),
        # a few requests gathered by a server, alternating full and local attention
        dict(name="encode_few", kind="encode", width="base", prec="bf16", layers=4, local=True, B=7, lo=19, hi=160),
        # a small batch of documents through the wide encoder, local layers
        dict(name="encode_mid", kind="encode", width="large", prec="bf16", layers=3, local=True, B=8, lo=64, hi=512),
        # the throughput shape of the benchmark: 64 rows of up to 512 tokens
        dict(name="encode_bulk", kind="encode", width="base", prec="bf16", layers=3, local=False, B=64, lo=64, hi=512),
        # long documents, full attention
        dict(name="encode_long", kind="encode", width="base", prec="bf16", layers=2, local=False, B=4, lo=4096, hi=8192),
        # the wide encoder with fp8 weights, 32 rows of up to 1024 tokens
        dict(name="encode_fp8", kind="encode", width="large", prec="fp8", layers=2, local=False, B=32, lo=256, hi=1024),
        # the fp32 mode, for callers who check results against the CPU forward
        dict(name="encode_fp32", kind="encode", width="base", prec="fp32", layers=2, local=True, B=5, lo=30, hi=200),
        # typed questions over shared documents: the decision head dominates
        dict(name="decide", kind="shared", width="base", prec="bf16", layers=2, local=False, B=12, lo=40, hi=300, questions=8),
        # the FFN product of a BERT-style layer on a ragged row count
        dict(name="gemm_gelu", kind="gemm", M=1501, N=3072, K=768, act=1, dtype="bf16"),
        # attention of a padded batch with a sliding window
        dict(name="attn_local", kind="attn", B=8, L=777, H=12, window=64, lo=200, hi=777, dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        kind = rng.choice(["encode"] * 5 + ["forward", "shared", "gemm", "attn"])
        if kind == "gemm":
            c = dict(kind=kind, M=_log(rng, 3, 20000), N=rng.choice([256, 768, 1024, 2304, 3072, 4096]),
                     K=rng.choice([768, 1024, 3072]), act=rng.choice([0, 1, 2]), dtype=rng.choice(["bf16", "bf16", "bf16", "fp32"]))
        elif kind == "attn":
            L = _log(rng, 16, 4096)
            c = dict(kind=kind, B=_log(rng, 1, 32), L=L, H=rng.choice([12, 16]), window=rng.choice([0, 64, 64]),
                     lo=rng.randint(max(1, L // 4), L), hi=L, dtype=rng.choice(["bf16", "bf16", "bf16", "fp32"]))
        else:
            prec = rng.choice(["bf16"] * 4 + ["fp8", "fp32"])
            width = "large" if prec == "fp8" else rng.choice(["base", "large"])
            hi = _log(rng, 9, 8192 if kind == "encode" else 700)
            B = _log(rng, 1, 64 if kind == "encode" else 24)
            layers = rng.choice([2, 3, 4]) if kind == "encode" else 2
            lo = rng.randint(max(1, hi // 8), hi)
            c = dict(kind=kind, width=width, prec=prec, layers=layers, local=rng.choice([False, True]), B=B, lo=lo, hi=hi)
            if kind == "shared":
                c["questions"] = rng.randint(1, 8)
        # no more than the largest listed case; the fp32 mode is for checks on small batches
        small = "fp32" in (c.get("prec"), c.get("dtype"))
        if work(c)["flops"] <= (4e10 if small else 1.4e12) and _tokens(c) <= 26000:
            return c


# ------------------------------------------------------------------ sizes --
def _lengths(case):
    B, lo, hi = case["B"], case["lo"], case["hi"]
    return [lo + round((hi - lo) * (i + 0.5) / B) for i in range(B)] if B > 1 else [hi]


def _tokens(case):
    return case["M"] if case["kind"] == "gemm" else case["B"] * case["L"] if case["kind"] == "attn" else sum(_lengths(case))


def _windows(case):
    """Window of each layer: 0 full, else |i - j| <= LOCAL / 2 (one full layer in three)."""
    return [LOCAL // 2 if case["local"] and i % 3 else 0 for i in range(case["layers"])]


def _pairs(n, m, w):
    """(query, key) pairs of n queries over m keys under a window."""
    if not w:
        return n * m
    i = np.arange(n)
    return int(np.maximum(np.minimum(i + w, m - 1) - np.maximum(i - w, 0) + 1, 0).sum())


def work(case):
    k = case["kind"]
    if k == "gemm":
        M, N, K, es = case["M"], case["N"], case["K"], 2 if case["dtype"] == "bf16" else 4
        return {"bytes": es * (M * K + N * K + M * N) + 4 * N, "flops": 2 * M * N * K}
    if k == "attn":
        B, L, D, es = case["B"], case["L"], case["H"] * 64, 2 if case["dtype"] == "bf16" else 4
        pairs = sum(_pairs(L, n, case["window"]) for n in _lengths(case))
        return {"bytes": es * 4 * B * L * D, "flops": 4 * D * pairs}
    w = WIDTHS[case["width"]]
    D, F, lens = w["hidden_size"], w["intermediate_size"], _lengths(case)
    T = sum(lens)
    mats = 4 * D * D + 3 * D * F
    es = {"fp32": 4, "bf16": 2, "fp8": 1}[case["prec"]]
    flops = sum(2 * T * mats + 4 * D * sum(_pairs(n, n, win) for n in lens) for win in _windows(case))
    nbytes = case["layers"] * mats * es + T * D * (4 if case["prec"] == "fp32" else 2)
    if k == "encode":
        return {"bytes": nbytes + T * (4 + 4 * D), "flops": flops}
    # the decision head: two biased layers over the rows (per sequence and type
    # of question where sequences are shared), the scorer per marker
    rows, types = case["B"], 1
    if k == "shared":
        rows, types = case["B"] * case["questions"], min(3, case["questions"])
    hmats = 12 * D * D
    flops += HEADS * types * (2 * T * hmats + 4 * D * sum(n * n for n in lens)) + rows * (K_MAX * 2 * D * D + 512 * (D + 4))
    nbytes += HEADS * hmats * (4 if case["prec"] == "fp32" else 2) + 4 * (D * D + 256 * (D + 4)) + rows * (K_MAX * 13 + 8 * N_ACT)
    return {"bytes": nbytes, "flops": flops}


# ---------------------------------------------------------------- weights --
def _bf16(x):
    return x.to(torch.bfloat16).to(torch.float32)


def _weights(width, layers, device="cuda"):
    """fp32 tensors of a DecisionModel, N(0, 0.02) rounded to bf16 (what a bf16
    checkpoint holds), norm gains around 1."""
    w = WIDTHS[width]
    D, F = w["hidden_size"], w["intermediate_size"]
    g = torch.Generator(device=device).manual_seed(1234 + D)

    def n(*s):
        return _bf16(torch.randn(*s, generator=g, device=device) * 0.02)

    def gain(d):
        return 1 + 0.05 * torch.randn(d, generator=g, device=device)

    t = {"encoder.embeddings.tok_embeddings.weight": n(VOCAB, D), "encoder.embeddings.norm.weight": gain(D)}
    for i in range(layers):
        p = f"encoder.layers.{i}."
        if i > 0:
            t[p + "attn_norm.weight"] = gain(D)
        t[p + "attn.Wqkv.weight"], t[p + "attn.Wo.weight"] = n(3 * D, D), n(D, D)
        t[p + "mlp_norm.weight"] = gain(D)
        t[p + "mlp.Wi.weight"], t[p + "mlp.Wo.weight"] = n(2 * F, D), n(D, F)
    t["encoder.final_norm.weight"] = gain(D)
    t["type_emb.weight"] = n(3, D)
    for i in range(HEADS):
        p = f"head.layers.{i}."
        for j in ("norm1", "norm2"):
            t[p + j + ".weight"], t[p + j + ".bias"] = gain(D), n(D)
        t[p + "self_attn.in_proj_weight"], t[p + "self_attn.in_proj_bias"] = n(3 * D, D), n(3 * D)
        t[p + "self_attn.out_proj.weight"], t[p + "self_attn.out_proj.bias"] = n(D, D), n(D)
        t[p + "linear1.weight"], t[p + "linear1.bias"] = n(4 * D, D), n(4 * D)
        t[p + "linear2.weight"], t[p + "linear2.bias"] = n(D, 4 * D), n(D)
    t["scorer.0.weight"], t["scorer.0.bias"] = gain(D), n(D)
    t["scorer.1.weight"], t["scorer.1.bias"] = n(D, D), n(D)
    t["scorer.3.weight"], t["scorer.3.bias"] = n(1, D), n(1)
    t["act_head.0.weight"], t["act_head.0.bias"] = n(256, D + 4), n(256)
    t["act_head.2.weight"], t["act_head.2.bias"] = n(N_ACT, 256), n(N_ACT)
    return t


@functools.lru_cache(maxsize=1)
def _model(width, layers, prec, local):
    t = _weights(width, layers)
    w = {k: v.cpu().numpy() for k, v in t.items()}
    types = ["sliding_attention" if local and i % 3 else "full_attention" for i in range(layers)]
    cfg = dict(WIDTHS[width], num_hidden_layers=layers, vocab_size=VOCAB, max_position_embeddings=MAX_POS, norm_eps=EPS,
               local_attention=LOCAL, layer_types=types, rope_theta_full=THETA, rope_theta_sliding=10000.0,
               head_layers=HEADS, n_act=N_ACT)
    return sj.Model(w, cfg, precision=PREC[prec])


# ----------------------------------------------------------------- inputs --
def _batch(case, seed):
    """Row lengths (in the seed's order) and token ids of each row."""
    rng = np.random.default_rng(seed)
    lens = rng.permutation(_lengths(case))
    return lens, [rng.integers(0, VOCAB, size=n) for n in lens]


def _host(case, seed):
    """Padded ids and mask [B, L], and one question per row (forward) or
    ``questions`` per sequence (shared): row_seq, marker_pos, marker_mask, qtype."""
    lens, rows = _batch(case, seed)
    L = max(case["hi"], int(lens.max()))
    ids, mask = np.zeros((len(rows), L), np.int64), np.zeros((len(rows), L), np.int64)
    for b, r in enumerate(rows):
        ids[b, :len(r)], mask[b, :len(r)] = r, 1
    rng = np.random.default_rng([seed, 1])
    row_seq = np.repeat(np.arange(len(rows)), case.get("questions", 1)).astype(np.int32)
    # the types in turn, so that the number of distinct ones per sequence is the case's
    qt = (np.arange(len(row_seq)) % 3).astype(np.int64)
    mp, mm = np.zeros((len(qt), K_MAX), np.int64), np.zeros((len(qt), K_MAX), np.uint8)
    for i, q in enumerate(qt):
        n = int(lens[row_seq[i]])
        lo, hi = MARKERS[int(q)]
        k = min(lo + 5 * i % (hi - lo + 1), max(case["lo"] - 1, 1))
        pos = rng.choice(np.arange(min(1, n - 1), max(n, 1)), size=k, replace=False)
        mp[i, :k], mm[i, :k] = np.sort(pos), 1
    return ids, mask, row_seq, mp, mm, qt


def _device_values(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32

    def r(*s):
        return torch.randn(*s, generator=g, device="cuda")

    if case["kind"] == "gemm":
        M, N, K = case["M"], case["N"], case["K"]
        return r(M, K).to(dt), (r(N, K) * 0.02).to(dt), r(N) * 0.02
    qkv = r(case["B"], case["L"], 3, case["H"], 64).to(dt)
    lens = np.random.default_rng(seed).permutation(_lengths(case)).astype(np.int32)
    return qkv, torch.from_numpy(lens).cuda()


def prepare(case, seed):
    k = case["kind"]
    st = {"case": case}
    if k in ("gemm", "attn"):
        st["lib"] = sj.lib()
        st["in"] = _device_values(case, seed)
        x = st["in"][0]
        shape = (case["M"], case["N"]) if k == "gemm" else (case["B"], case["L"], case["H"] * 64)
        st["out"] = torch.empty(shape, dtype=x.dtype, device="cuda")
        return st
    st["model"] = _model(case["width"], case["layers"], case["prec"], case["local"])
    if k == "encode":
        lens, rows = _batch(case, seed)
        st["lens"] = lens.astype(np.int32)
        st["ids"] = torch.from_numpy(np.concatenate(rows).astype(np.int32)).cuda()
        st["out"] = torch.empty(int(lens.sum()), WIDTHS[case["width"]]["hidden_size"], dtype=torch.float32, device="cuda")
    else:
        st["in"] = _host(case, seed)
    return st


def run(st):
    case = st["case"]
    k = case["kind"]
    if k == "encode":
        st["model"].encode_device(st["ids"].data_ptr(), st["lens"], st["out"].data_ptr())
        return st["out"]
    if k == "forward":
        ids, mask, _, mp, mm, qt = st["in"]
        logits, act = st["model"].forward(ids, mask, mp, mm, qt)
        return logits, act, logits[mm != 0]  # the options' own logits: what calibration reads next
    if k == "shared":
        ids, mask, row_seq, mp, mm, qt = st["in"]
        logits, act = st["model"].forward_shared(ids, mask, row_seq, mp, mm, qt)
        return logits, act, logits[mm != 0]
    p = [ctypes.c_void_p(x.data_ptr()) for x in (*st["in"], st["out"])]
    dt = sj.SJH_BF16 if case["dtype"] == "bf16" else sj.SJH_F32
    if k == "gemm":
        sj.check(st["lib"].sjh_gemm(p[0], p[1], p[2], p[3], case["M"], case["N"], case["K"], case["act"], dt, None))
    else:
        sj.check(st["lib"].sjh_attn(p[0], p[1], p[2], case["B"], case["L"], case["H"], 64, case["window"], dt, None))
    return st["out"]


# ------------------------------------------------------------------ exact --
def _ln64(x, w, b=None):
    m = x.mean(-1, keepdim=True)
    y = (x - m) / torch.sqrt(((x - m) ** 2).mean(-1, keepdim=True) + EPS) * w
    return y if b is None else y + b


def _gelu64(x):
    return 0.5 * x * (1 + torch.erf(x / math.sqrt(2.0)))


def _attn64(q, k, v, window):
    """[n, H, 64] queries over [m, H, 64] keys, head by head."""
    n, m = q.shape[0], k.shape[0]
    out = torch.empty_like(q)
    far = None
    if window:
        far = (torch.arange(n, device=q.device)[:, None] - torch.arange(m, device=q.device)[None]).abs() > window
    for h in range(q.shape[1]):
        s = q[:, h] @ k[:, h].t().contiguous() / 8.0
        if far is not None:
            s = s.masked_fill(far, -math.inf)
            p = torch.softmax(s, -1).nan_to_num(0.0)  # a query past the last key's window reads nothing
        else:
            p = torch.softmax(s, -1)
        out[:, h] = p @ v[:, h].contiguous()
    return out


def _rope64(x, theta):
    n, half = x.shape[0], 32
    inv = theta ** (-2.0 * torch.arange(half, device=x.device, dtype=torch.float64) / 64)
    a = torch.arange(n, device=x.device, dtype=torch.float64)[:, None] * inv[None]
    c, s = a.cos()[:, None], a.sin()[:, None]
    x1, x2 = x[..., :half], x[..., half:]
    return torch.cat([x1 * c - x2 * s, x2 * c + x1 * s], -1)


def _fp8(w):
    """Rows as e4m3 codes times one fp32 scale each (absmax / 448)."""
    sc = w.abs().amax(1) / 448.0
    sc = torch.where(sc == 0, torch.ones_like(sc), sc)
    return (w / sc[:, None]).to(torch.float8_e4m3fn).to(torch.float64) * sc.double()[:, None]


def _encode64(case, t, rows):
    D = WIDTHS[case["width"]]["hidden_size"]
    F, H = WIDTHS[case["width"]]["intermediate_size"], D // 64
    mat = _fp8 if case["prec"] == "fp8" else (lambda x: x.double())
    lens = [len(r) for r in rows]
    ids = torch.from_numpy(np.concatenate(rows)).cuda()
    x = _ln64(t["encoder.embeddings.tok_embeddings.weight"][ids].double(), t["encoder.embeddings.norm.weight"].double())
    for i, win in enumerate(_windows(case)):
        p = f"encoder.layers.{i}."
        y = _ln64(x, t[p + "attn_norm.weight"].double()) if i else x
        qkv = (y @ mat(t[p + "attn.Wqkv.weight"]).t()).view(-1, 3, H, 64)
        theta = 10000.0 if win else THETA
        o = [_attn64(_rope64(s[:, 0], theta), _rope64(s[:, 1], theta), s[:, 2], win) for s in qkv.split(lens)]
        x = x + torch.cat(o).reshape(-1, D) @ mat(t[p + "attn.Wo.weight"]).t()
        u = _ln64(x, t[p + "mlp_norm.weight"].double()) @ mat(t[p + "mlp.Wi.weight"]).t()
        x = x + (_gelu64(u[:, :F]) * u[:, F:]) @ mat(t[p + "mlp.Wo.weight"]).t()
    return list(_ln64(x, t["encoder.final_norm.weight"].double()).split(lens))


def _decide64(t, seqs, row_seq, mp, mm, qt):
    D = seqs[0].shape[1]
    t = {k: v.double() for k, v in t.items() if not k.startswith("encoder.")}
    done, logits, act = {}, [], []
    for i, q in enumerate(qt):
        u = int(row_seq[i])
        if (u, int(q)) not in done:
            h = seqs[u] + t["type_emb.weight"][int(q)]
            for li in range(HEADS):
                g = lambda n: t[f"head.layers.{li}." + n]  # noqa: E731
                y = _ln64(h, g("norm1.weight"), g("norm1.bias"))
                s = (y @ g("self_attn.in_proj_weight").t() + g("self_attn.in_proj_bias")).view(-1, 3, D // 64, 64)
                o = _attn64(s[:, 0], s[:, 1], s[:, 2], 0).reshape(-1, D)
                h = h + o @ g("self_attn.out_proj.weight").t() + g("self_attn.out_proj.bias")
                y = _ln64(h, g("norm2.weight"), g("norm2.bias"))
                f = torch.relu(y @ g("linear1.weight").t() + g("linear1.bias"))
                h = h + f @ g("linear2.weight").t() + g("linear2.bias")
            done[u, int(q)] = h
        h = done[u, int(q)]
        s = _ln64(h[torch.from_numpy(mp[i]).cuda()], t["scorer.0.weight"], t["scorer.0.bias"])
        s = _gelu64(s @ t["scorer.1.weight"].t() + t["scorer.1.bias"])
        on = torch.from_numpy(mm[i]).cuda().bool()
        lg = torch.where(on, (s @ t["scorer.3.weight"].t() + t["scorer.3.bias"])[:, 0], -1e4)
        p = torch.softmax(lg, 0)
        top = p.sort(descending=True).values
        kf = max(2.0, float(on.sum()))
        ent = -(p * p.clamp(min=1e-9).log()).sum() / math.log(kf)
        x = torch.cat([h[0], torch.stack([top[0], top[0] - top[1], ent, torch.full_like(ent, kf / 255.0)])])
        a = _gelu64(t["act_head.0.weight"] @ x + t["act_head.0.bias"])
        logits.append(lg)
        act.append(torch.softmax(t["act_head.2.weight"] @ a + t["act_head.2.bias"], 0))
    return torch.stack(logits), torch.stack(act)


def exact(case, seed):
    k = case["kind"]
    if k == "gemm":
        a, w, b = (x.double() for x in _device_values(case, seed))
        c = a @ w.t() + b
        return _gelu64(c) if case["act"] == 1 else torch.relu(c) if case["act"] == 2 else c
    if k == "attn":
        qkv, lens = _device_values(case, seed)
        out = []
        for b, n in enumerate(lens.tolist()):
            x = qkv[b].double()
            out.append(_attn64(x[:, 0], x[:n, 1], x[:n, 2], case["window"]))
        return torch.stack(out).reshape(case["B"], case["L"], -1)
    t = _weights(case["width"], case["layers"])
    if k == "encode":
        return torch.cat(_encode64(case, t, _batch(case, seed)[1]))
    ids, mask, row_seq, mp, mm, qt = _host(case, seed)
    rows = [r[:int(n)] for r, n in zip(ids, mask.sum(1))]
    logits, act = _decide64(t, _encode64(case, t, rows), row_seq, mp, mm, qt)
    return logits, act, logits[torch.from_numpy(mm).cuda() != 0]


def tolerance(case):
    """About four times the distance of the path from ``exact`` as measured: bf16
    products and attention lie 1.7e-3 to 2.1e-3 from it (one rounding of the
    output), hidden states of two to four layers 0.5e-3 to 1.7e-3, the decision
    head's logits 0.9e-3 to 1.8e-3, everything in fp32 up to 2e-6."""
    return {"rel": 1e-5} if "fp32" in (case.get("prec"), case.get("dtype")) else {"rel": 8e-3}
