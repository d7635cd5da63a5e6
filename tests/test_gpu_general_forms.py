"""The operand forms and tile edges of the general attention kernel, against float64.

The kernel picks its matrix instructions from the operand types (bf16 or fp16 scores, fp32
scores; P-hat with bf16 V, anything with fp32), its instance from head_dim (64, 96, 128, 192,
256) and runs key tiles in groups of 128 keys of two 64-key halves.  Each case sits at an edge
of those, with unquantized P (no code to flip), so that a dense float64 softmax is the
reference and the bound follows from fp32 arithmetic: a score is off by at most
e = (D + 4) 2^-24 scale sum_d |q_d k_d|, P by a factor exp(2 e) (its own and the maximum's
error) and 4 ulp of exp, the two sums over Lk keys by Lk 2^-24 each, so
|o - ref| <= (2 e + (2 Lk + 8) 2^-24) 2 max |V|.
"""

from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

U = 2.0**-24


def _general(q, k, v, T, *, causal=True, quant_p=False, **kw):
    from faquant_amd import _ops

    out = torch.full(q.shape, float("nan"), device=q.device, dtype=torch.float32)
    _ops.attention_general(q, k, v, key_tile=T, causal=causal, scale=q.shape[-1] ** -0.5, quant_p=quant_p,
                           p_levels="123", norm_same=quant_p, out=out, **kw)
    return out


def _dense(q, k, v, causal):
    G = q.shape[1] // k.shape[1]
    qd, kd, vd = q.double(), k.double().repeat_interleave(G, 1), v.double().repeat_interleave(G, 1)
    scale = q.shape[-1] ** -0.5
    s = torch.matmul(qd, kd.transpose(-1, -2).contiguous()) * scale
    mag = torch.matmul(qd.abs(), kd.abs().transpose(-1, -2).contiguous()) * scale
    Lq, Lk = s.shape[-2:]
    if causal:
        seen = torch.arange(Lk, device=s.device)[None, :] <= torch.arange(Lq, device=s.device)[:, None] + Lk - Lq
        s = s.masked_fill(~seen, float("-inf"))
    p = torch.nan_to_num(torch.softmax(s, -1))  # rows that see no key output zero
    e = (q.shape[-1] + 4) * U * mag.amax()
    bound = (2 * e + (2 * Lk + 8) * U) * 2 * vd.abs().amax()
    return torch.matmul(p, vd), bound


DTYPES = {"b": torch.bfloat16, "h": torch.float16, "f": torch.float32}


@pytest.mark.parametrize("types", ["bbb", "hhh", "fff", "bbf", "hhb", "ffb", "bfh", "hbf"])
@pytest.mark.parametrize("D,T,Lq,Lk,Hq,Hkv", [
    (1, 64, 5, 9, 1, 1), (32, 63, 33, 70, 4, 1), (33, 65, 40, 130, 2, 2), (64, 128, 129, 129, 8, 2),
    (65, 127, 31, 200, 2, 1), (96, 129, 64, 257, 3, 3), (97, 16, 20, 50, 4, 4), (128, 256, 130, 300, 4, 2),
    (129, 1, 3, 6, 2, 1), (192, 128, 65, 140, 1, 1), (193, 100, 30, 101, 2, 2), (256, 1024, 70, 1100, 2, 1)])
def test_operand_forms_and_edges(dev, types, D, T, Lq, Lk, Hq, Hkv):
    g = torch.Generator(device="cpu").manual_seed(D * 7 + T)
    q, k, v = (torch.randn(2, h, n, D, generator=g).to(dev, DTYPES[t])
               for t, h, n in zip(types, (Hq, Hkv, Hkv), (Lq, Lk, Lk)))
    got = _general(q, k, v, T)
    ref, bound = _dense(q, k, v, True)
    err = (got.double() - ref).abs().max()
    print(f"[general form] {types} D{D} T{T}: error {float(err):.2e}, bound {float(bound):.2e}", flush=True)
    assert err <= bound  # a NaN left in out fails too


@pytest.mark.parametrize("types", ["bbb", "hhh", "fff"])
def test_unaligned_and_strided_operands(dev, types):
    """Rows that start off 16-byte alignment, odd row strides and a [B, L, H, D] layout give the
    bits of the contiguous operands (the loads differ, the arithmetic does not)."""
    g = torch.Generator(device="cpu").manual_seed(3)
    dt = DTYPES[types[0]]
    q, k, v = (torch.randn(1, h, 90, 72, generator=g).to(dev, dt) for h in (4, 2, 2))
    want = _general(q, k, v, 80)
    wide = [torch.randn(1, t.shape[1], 90, 75, generator=g).to(dev, dt) for t in (q, k, v)]
    for w, t in zip(wide, (q, k, v)):
        w[..., 1:73] = t
    assert torch.equal(_general(*(w[..., 1:73] for w in wide), 80), want)
    blhd = [t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v)]
    assert torch.equal(_general(*blhd, 80), want)


@pytest.mark.parametrize("types", ["bbb", "fff"])
def test_non_finite_scores(dev, types):
    """A score that is not finite gets P = 0 (the simulator's isfinite select): a NaN score
    drops its key; a +inf one becomes the maximum and drops the whole tile sequence so far."""
    g = torch.Generator(device="cpu").manual_seed(5)
    dt = DTYPES[types[0]]
    q, k, v = (torch.randn(1, 1, 40, 64, generator=g).to(dev, dt) for _ in range(3))
    k[0, 0, 7, 3] = float("nan")
    got = _general(q, k, v, 64, causal=False)
    keep = [i for i in range(40) if i != 7]
    ref, bound = _dense(q, k[:, :, keep], v[:, :, keep], False)
    assert (got.double() - ref).abs().max() <= bound
    k[0, 0, 7] = 0
    k[0, 0, 7, 3] = float("inf")
    q[..., 3] = q[..., 3].abs() + 0.5  # every score of key 7 is +inf
    assert not torch.any(_general(q, k, v, 64, causal=False))
