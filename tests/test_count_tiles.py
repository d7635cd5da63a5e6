"""The stats counters' closed form (count_tiles) against the simulator's schedule replayed tile
by tile (sfa:623-697, 886-908), over random lengths, chunks and flags."""

from __future__ import annotations

import random

import pytest

pytest.importorskip("torch")


def _replay(stats, *, batch, query_heads, query_length, key_length, head_dim, query_chunk, key_chunk, causal,
            skip_fully_masked, qk_quant, pv_quant, qk_group, pv_group):
    from faquant_amd.simulated_flash_attention import _record

    full, done = query_length // query_chunk, 0
    for q0, rows, tiles in ((0, query_chunk, full), (full * query_chunk, query_length - full * query_chunk, 1)):
        if rows == 0 or tiles == 0:
            continue
        if qk_quant:
            _record(stats, "q", head_dim, batch * query_heads * rows * head_dim, qk_group, tiles)
        for k0 in range(0, key_length, key_chunk):
            width = min(key_chunk, key_length - k0)
            for t in range(tiles):
                last_row = q0 + (t + 1) * rows - 1
                if skip_fully_masked and causal and k0 > last_row + key_length - query_length:
                    continue
                if qk_quant:
                    _record(stats, "k", head_dim, batch * query_heads * width * head_dim, qk_group, 1)
                if pv_quant:
                    _record(stats, "p", width, batch * query_heads * rows * width, pv_group, 1)
                    _record(stats, "v", head_dim, batch * query_heads * width * head_dim, pv_group, 1)
                done += 1
    stats["calls"] += 1
    for name, quantized in (("qk", qk_quant), ("pv", pv_quant)):
        stats[f"{name}_tiles"] += done
        if quantized:
            stats[f"{name}_quantized_tiles"] += done


@pytest.mark.parametrize("seed", range(8))
def test_closed_form_equals_the_schedule(seed):
    from faquant_amd.simulated_flash_attention import count_tiles, new_simulated_attention_stats

    r = random.Random(seed)
    for _ in range(60):
        key_length = r.randint(1, 700)
        kw = dict(batch=r.randint(1, 2), query_heads=r.choice([1, 4]), key_length=key_length, head_dim=r.choice([64, 72]),
                  query_length=r.choice([1, key_length, r.randint(1, 900)]), query_chunk=r.choice([1, 7, 64, 256, 1000]),
                  key_chunk=r.choice([1, 37, 64, 100, 128, 2000]), causal=r.random() < 0.7,
                  skip_fully_masked=r.random() < 0.7, qk_quant=r.random() < 0.7, pv_quant=r.random() < 0.7,
                  qk_group=64, pv_group=64)
        got, want = new_simulated_attention_stats(), new_simulated_attention_stats()
        count_tiles(got, **kw)
        _replay(want, **kw)
        assert got == want, kw
