"""Short batches (up to 256 rows): the products that keep most of K in flight and
the residual products that cut K over the waves of a workgroup.

Every row is held to the oracle within the bf16 tolerance of the hidden states,
and has the same bits alone as in a batch that fills the range (whose tiles
outnumber the CUs and take a shorter ring)."""
import numpy as np
import pytest

import snapjudge_amd as sj
from snapjudge_amd import synth

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

WIDTHS = {256: (4, 320), 512: (8, 768), 768: (12, 1152), 1024: (16, 2624)}


def model(D, seed, **kw):
    H, F = WIDTHS[D]
    rl, enc, w = synth.make_model(hidden_size=D, num_hidden_layers=2, num_attention_heads=H, intermediate_size=F,
                                  vocab_size=1024, theta_full=160000.0, store="BF16", seed=seed, **kw)
    return synth.flat_cfg(rl, enc), w


# one to four groups of K in the load ring; one row, the edges of a 32-row tile,
# the last batch of the range
@pytest.mark.parametrize("D", [256, 512, 768, 1024])
@pytest.mark.parametrize("lens", [[1], [32], [33], [65, 32], [96, 1], [127], [64, 64], [130, 126]])
def test_short_rows_keep_their_bits(orc, D, lens):
    print(f"short rows D={D} lens={lens}", flush=True)
    cfg, w = model(D, seed=3 + D)
    m = sj.Model(w, cfg, precision=sj.SJH_PREC_BF16)
    fill = [256 - sum(lens)] if sum(lens) < 256 else []
    ids, mask, _ = synth.batch_with_lens(lens + fill, max(lens + fill), 1024, seed=5)
    n = len(lens)
    short = m.encode(ids[:n, :max(lens)], mask[:n, :max(lens)])
    full = m.encode(ids, mask)
    om = orc.model(w, cfg)
    for b, k in enumerate(lens):
        ref = om.encode(ids[b:b + 1, :k], mask[b:b + 1, :k])[0]
        assert float(np.abs(short[b, :k] - ref).max()) <= 2e-2
        assert np.array_equal(short[b, :k], full[b, :k]), f"row {b}"
    m.close()


@pytest.mark.parametrize("D,lens", [(256, [33]), (768, [97, 31]), (1024, [70]), (1024, [256])])
def test_short_fp8_rows(orc, D, lens):
    # the fp8 kernels of the same sizes, against the oracle on the dequantized
    # weights; the decision head's layers run on the bf16 ones
    print(f"short fp8 rows D={D} lens={lens}", flush=True)
    cfg, w = model(D, seed=11 + D)
    m = sj.Model(w, cfg, precision=sj.SJH_PREC_FP8W)
    ids, mask, n = synth.batch_with_lens(lens, max(lens), 1024, seed=6)
    om = orc.model(sj.fp8_dequantized(w), cfg)
    h, ref = m.encode(ids, mask), om.encode(ids, mask)
    assert float(np.abs(h - ref)[mask.astype(bool)].max()) <= 2e-2
    # the same bits in a batch that fills the range, where the products of more than
    # two rounds of tiles go to the tiled kernels
    if sum(lens) < 256:
        fids, fmask, _ = synth.batch_with_lens(lens + [256 - sum(lens)], 256 - sum(lens), 1024, seed=6)
        fids[:len(lens), :ids.shape[1]] = ids
        full = m.encode(fids, fmask)
        for b, k in enumerate(lens):
            assert np.array_equal(h[b, :k], full[b, :k]), f"row {b}"
    mp, mm, qt = synth.make_markers(n, 4, [(0, 4), (2, 2)][:len(lens)], seed=7)
    logits, act = m.forward(ids, mask, mp, mm, qt)
    rl, ra = om.forward(ids, mask, mp, mm, qt)
    for b in range(len(lens)):
        k = int(mm[b].sum())
        p, r = orc.calibrated_probs(logits[b, :k], 1.0), orc.calibrated_probs(rl[b, :k], 1.0)
        assert float(np.abs(p - r).max()) <= 5e-3
    assert float(np.abs(act - ra).max()) <= 5e-3
    m.close()


@pytest.mark.parametrize("prec", [sj.SJH_PREC_BF16, sj.SJH_PREC_FP8W])
def test_short_batch_beside_a_full_scratch_array(prec):
    # 256 rows of this width leave no room for the residual stream in the fixed
    # array: the batch still runs there, on the caller's rows, with the same bits
    # (fp8 weights too: its residual products keep their K slices); rows past the
    # batch, of which a launch has some, are not the caller's
    rl, enc, w = synth.make_model(hidden_size=1664, num_hidden_layers=1, num_attention_heads=26,
                                  intermediate_size=1024, vocab_size=512, store="BF16", seed=23)
    m = sj.Model(w, synth.flat_cfg(rl, enc), precision=prec)
    for lens in ([256], [150, 101], [100, 41]):
        ids, _, n = synth.batch_with_lens(lens, max(lens), 512, seed=8)
        print(f"full scratch array prec={prec} lens={lens}", flush=True)
        d_ids = torch.from_numpy(np.concatenate([ids[b, :k] for b, k in enumerate(lens)]).astype(np.int32)).cuda()
        outs = []
        for fn in (m.encode_device, m.encode_device_noalloc):
            out = torch.full((sum(lens) + 64, 1664), float("nan"), dtype=torch.float32, device="cuda")
            fn(d_ids.data_ptr(), np.asarray(lens, np.int32), out.data_ptr(), torch.cuda.current_stream().cuda_stream)
            torch.cuda.synchronize()
            assert bool(torch.isnan(out[sum(lens):]).all())
            outs.append(out[:sum(lens)].cpu().numpy())
        assert np.isfinite(outs[0]).all() and np.array_equal(outs[0], outs[1])
    m.close()
