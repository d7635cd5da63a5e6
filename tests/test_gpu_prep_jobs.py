"""The operand prologues of an attention call in one launch (faq_operand_prep_jobs) against the
single entries, bit for bit: row jobs of one and several blocks, ragged tails, packed rows at an
offset, V^T with and without natural rows, every level form, and lists that run job by job
(fp32, more row jobs than one launch takes)."""

from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("B,H,L,lv,had", [(1, 1, 1, "123", 0), (2, 3, 31, "12", 64), (1, 8, 64, "13", 128),
                                          (3, 2, 65, "123", 64), (1, 2, 129, None, 0), (2, 1, 1000, "123", 128)])
def test_jobs_equal_single_entries(dev, dtype, B, H, L, lv, had):
    from faquant_amd import _ops

    g = torch.Generator(device="cpu").manual_seed(L)
    dt, bf = getattr(torch, dtype), torch.bfloat16
    q = torch.randn(B, 2 * H, 5, 128, generator=g).to(dev, dt)
    k = torch.randn(B, L, H, 128, generator=g).to(dev, dt).transpose(1, 2)
    v = torch.randn(B, H, L, 128, generator=g).to(dev, dt)
    k[0, 0, 0, 3] = float("nan")
    offset, smooth = torch.randn(H, 128, generator=g).to(dev), torch.rand(H, 128, generator=g).to(dev) + 0.5
    k_kw = dict(levels=lv, hadamard=had, key_offset=offset, smooth=smooth, smooth_divide=True, round_dtype=bf)
    q_kw = dict(levels="12", hadamard=had, round_dtype=bf)
    cap = torch.full((B, H, L + 7, 128), 5.0, device=dev, dtype=bf)
    kb, qb, vb = cap[:, :, :L], torch.empty_like(q, dtype=bf), torch.empty(B, H, L, 128, device=dev, dtype=bf)
    vt = torch.full((B, H, 128, _ops._pad_keys(L)), 3.0, device=dev, dtype=bf)
    _ops.operand_prep_jobs([_ops.prep_job(q, out=qb, **q_kw), _ops.prep_job(k, out=kb, **k_kw),
                            _ops.prep_job(v, levels=lv, out=vb, vt=vt)], dev)
    bits = lambda t: t.contiguous().view(torch.int16)  # noqa: E731  (NaN groups compare by their bits)
    assert torch.equal(bits(qb), bits(_ops.operand_prep(q, **q_kw)[0]))
    assert torch.equal(bits(kb), bits(_ops.operand_prep(k, **k_kw)[0]))
    assert torch.equal(bits(vb), bits(_ops.operand_prep(v, levels=lv)[0]))
    assert torch.equal(bits(vt), bits(_ops.operand_prep_vt(v, levels=lv)))
    assert torch.all(cap[:, :, L:] == 5.0)
    vt2 = torch.empty_like(vt)
    _ops.operand_prep_jobs([_ops.prep_job(v, levels=lv, vt=vt2)], dev)
    assert torch.equal(bits(vt2), bits(vt))
    if lv:
        one, many = (_ops.PackedHiF4KV(B, H, L + 9, dev, lv) for _ in range(2))
        _ops.pack_operand(k, out=one, start=4, **k_kw)
        jobs = [_ops.prep_job(k, packed=many, start=4, **k_kw)]
        jobs += [_ops.prep_job(q, out=torch.empty_like(qb), **q_kw) for _ in range(3)]  # four row jobs
        _ops.operand_prep_jobs(jobs, dev)
        few = _ops.PackedHiF4KV(B, H, L + 9, dev, lv)
        _ops.operand_prep_jobs([_ops.prep_job(k, packed=few, start=4, **k_kw)], dev)
        for p in (many, few):
            assert torch.equal(p.codes[:, :, 4:4 + L], one.codes[:, :, 4:4 + L])
            assert torch.equal(p.meta[:, :, 4:4 + L], one.meta[:, :, 4:4 + L])


def test_a_refused_call_leaves_the_caches_alone(dev):
    """K rows off 16-byte alignment are refused, and the module keeps the cache it had."""
    from faquant_amd.simulated_flash_attention import simulated_flash_attention_forward
    from tests.test_gpu_attention import module

    m = module()
    x = torch.randn(1, 1, 40, 128, device=dev).to(torch.bfloat16)
    simulated_flash_attention_forward(m, x, x, x, None)
    before = m.faquant_k_matmul_qdq_cache
    bad = torch.randn(1, 1, 41, 132, device=dev).to(torch.bfloat16)[..., 1:129]
    with pytest.raises(ValueError):
        simulated_flash_attention_forward(m, x, bad, bad, None)
    assert m.faquant_k_matmul_qdq_cache is before
