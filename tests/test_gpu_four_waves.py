"""The four-wave form of the attention kernel against the eight-wave one: the same operations in
the same order per row, so the same bits (outputs and denominators), at the edges of its
items (128 rows of 4, 2 or 1 heads), tiles and pairings, with and without key ranges."""

from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,Lq,Lk,causal,masked", [
    (1, 4, 1, 1, 1, True, False), (1, 4, 4, 127, 128, True, False), (2, 6, 3, 129, 129, True, False),
    (1, 32, 8, 1999, 1999, True, False), (1, 16, 1, 33, 300, True, False), (1, 5, 1, 300, 260, True, False),
    (3, 8, 2, 500, 500, False, False), (1, 40, 40, 700, 257, False, False), (1, 32, 8, 2300, 2300, True, False),
    (3, 8, 2, 390, 390, True, True), (2, 3, 3, 200, 700, True, True), (2, 4, 2, 70, 513, False, True)])
@pytest.mark.parametrize("quant_p,same,levels,out_levels,f32", [
    (True, True, "123", None, False), (True, False, "12", "123", False), (False, False, "13", None, True)])
def test_four_waves_equal_eight_waves(dev, monkeypatch, B, Hq, Hkv, Lq, Lk, causal, masked, quant_p, same, levels,
                                      out_levels, f32):
    from faquant_amd import _ops

    g = torch.Generator(device="cpu").manual_seed(Lq * 3 + Lk)
    q, k, v = (torch.randn(B, h, n, 128, generator=g).to(dev, torch.bfloat16)
               for h, n in ((Hq, Lq), (Hkv, Lk), (Hkv, Lk)))
    kh, _ = _ops.operand_prep(k, levels=levels)
    vt = _ops.operand_prep_vt(v, levels=levels)
    ranges = None
    if masked:
        mask = torch.rand(B, Lk, generator=g) > 0.1
        mask[0, : Lk // 3] = False
        ranges = _ops.attention_key_ranges(mask.to(dev), B, Lq, Lk, causal=causal)
    res = {}
    for waves in ("8", "4"):
        monkeypatch.setenv("FAQ_ATTN_WAVES", waves)
        out = torch.full((B, Lq, Hq, 128), float("nan"), device=dev, dtype=torch.float32 if f32 else torch.bfloat16)
        den = torch.full((B, Hq, Lq), float("nan"), device=dev)
        _ops.attention_fwd(q, kh, vt, Lk, causal=causal, scale=128**-0.5, quant_p=quant_p, p_levels=levels,
                           norm_same=same, out=out.transpose(1, 2), row_den=den, split=1, ranges=ranges,
                           out_levels=out_levels, q_prep=(64, levels))
        assert torch.isfinite(out).all()
        res[waves] = out, den
    assert torch.equal(res["4"][0], res["8"][0])
    assert torch.equal(res["4"][1], res["8"][1])
