"""The work this library is used for, as cases that can be timed and compared.

Each case is one call that a user's program makes through a public entry point: a prefill or
a decode step of a Qwen3 attention layer, a Wan2.2 self- or cross-attention, a quantized
Linear, the codec on a weight.  ``prepare`` makes what the program has in hand before that
call, ``run`` makes the call, ``exact`` computes the same result in plain float64 torch.

The HiF4 quantizer is part of the result: its scale and reciprocal are bf16 numbers and its
codes integers, so float64 restates its definition (the same bf16 roundings) and differs
from float32 only where a value lies within float32 rounding of a code boundary.
"""

from __future__ import annotations

import math
import os
import sys
from types import SimpleNamespace

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "faquant-public_amd"))

DEVICE = "cuda:0"
HIF4 = {"quant_format": "hif4", "bits": 4, "group_size": 64, "symmetric": True, "clip_ratio": 1.0}


def listed() -> list[dict]:
    return [
        # The headline workload: one Qwen3-8B layer's causal prefill of 32k tokens, from the
        # post-RoPE Q/K/V to the attention output (block Hadamard of 64, HiF4 Q/K/P/V).
        {"name": "qwen8b_prefill_32k", "kind": "prefill", "batch": 1, "hq": 32, "hkv": 8, "lq": 32768, "lk": 32768},
        # A prompt of ordinary length, not a multiple of any tile, as a chat request brings it.
        {"name": "qwen8b_prefill_1999", "kind": "prefill", "batch": 1, "hq": 32, "hkv": 8, "lq": 1999, "lk": 1999},
        # Batched evaluation (multiple-choice prompts): left-padded prompts of unequal length
        # with the 2-D mask that transformers passes to the attention backend.
        {"name": "qwen8b_batch_padded", "kind": "padded", "batch": 8, "hq": 32, "hkv": 8, "l": 777},
        # Wan2.2 DiT self-attention at 480p: 40 heads, every token sees every token.
        {"name": "wan480p_self", "kind": "wan", "heads": 40, "lq": 32760, "lk": 32760},
        # The cross-attention of the same block: the video tokens against 512 text tokens.
        {"name": "wan480p_cross", "kind": "wan", "heads": 40, "lq": 32760, "lk": 512},
        # One generated token over an 8k context: the smallest attention call, bf16 caches.
        {"name": "qwen8b_decode_8k", "kind": "decode", "batch": 1, "hq": 32, "hkv": 8, "l": 8150, "packed": False},
        # One generated token over a long context with the packed 4.5-bit K/V caches.
        {"name": "qwen8b_decode_128k_packed", "kind": "decode", "batch": 1, "hq": 32, "hkv": 8, "l": 131000,
         "packed": True},
        # down_proj of Qwen3-8B over a prefill of 4096 tokens with every activation step on: the
        # HiSQ rotation (blocks of 1024), the clamp, the companding and the HiF4 QDQ.
        {"name": "linear_prefill_4096", "kind": "linear", "rows": 4096, "k": 12288, "n": 4096, "rotation": 1024,
         "packed": False},
        # gate_proj of one generated token with the packed weight: the smallest Linear call.
        {"name": "linear_decode_1", "kind": "linear", "rows": 1, "k": 4096, "n": 12288, "rotation": 1024,
         "packed": True},
        # The key-chunk ablation of the simulator: the same attention with chunks of 64 keys.
        {"name": "ablation_chunk64", "kind": "ablation", "hq": 32, "hkv": 8, "l": 4096, "d": 128, "chunk": 64,
         "dtype": "bfloat16", "qk": True, "pv": True},
        # The PV-only ablation on fp32 activations: Q and K multiplied unquantized in fp32.
        {"name": "ablation_fp32_pv_only", "kind": "ablation", "hq": 16, "hkv": 8, "l": 2000, "d": 128, "chunk": 128,
         "dtype": "float32", "qk": False, "pv": True},
        # Quantizing a model: the codec over one down_proj weight.
        {"name": "codec_weight", "kind": "codec", "rows": 4096, "cols": 12288, "dtype": "bfloat16"},
    ]


def _log(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng) -> dict:
    kind = rng.choice(["prefill", "padded", "wan", "decode", "decode", "linear", "linear", "ablation", "codec"])
    if kind == "prefill":
        hq, hkv = rng.choice([(32, 8), (64, 8), (16, 8), (40, 8)])
        lq = _log(rng, 16, 12000)
        # a whole prompt, or the next chunk of one whose first part is already cached
        lk = lq if rng.random() < 0.6 else lq + _log(rng, 128, 12000)
        return {"kind": kind, "batch": rng.choice([1, 1, 2]), "hq": hq, "hkv": hkv, "lq": lq, "lk": lk}
    if kind == "padded":
        return {"kind": kind, "batch": rng.randint(2, 12), "hq": 32, "hkv": 8, "l": _log(rng, 64, 2500)}
    if kind == "wan":
        lq = _log(rng, 1000, 20000)
        return {"kind": kind, "heads": rng.choice([12, 24, 40]), "lq": lq, "lk": rng.choice([lq, 512, 257])}
    if kind == "decode":
        batch = rng.choice([1, 1, 1, 2, 4])
        hq, hkv = rng.choice([(32, 8), (64, 8), (16, 8)])
        length = _log(rng, 1000, 131000 // batch)
        # the caches hold length - 1 positions; one that is full to its capacity (a multiple of
        # 128) is copied into a larger one, which happens once in a thousand steps: not here
        if length % 128 == 1:
            length += 1
        return {"kind": kind, "batch": batch, "hq": hq, "hkv": hkv, "l": length, "packed": rng.random() < 0.5}
    if kind == "linear":
        k, n = rng.choice([(4096, 4096), (4096, 12288), (12288, 4096), (5120, 5120), (5120, 13824), (4096, 1024)])
        packed = rng.random() < 0.4
        rows = rng.randint(1, 4) if packed else _log(rng, 1, 8000)
        return {"kind": kind, "rows": rows, "k": k, "n": n, "rotation": rng.choice([0, 1024]), "packed": packed}
    if kind == "ablation":
        dtype = rng.choice(["bfloat16", "bfloat16", "float32", "float16"])
        qk, pv = rng.choice([(True, True), (True, True), (False, True), (True, False), (False, False)])
        hkv = rng.choice([2, 4, 8])
        return {"kind": kind, "hq": hkv * rng.choice([1, 2, 4]), "hkv": hkv, "l": _log(rng, 100, 3000),
                "d": rng.choice([64, 80, 96, 128, 128, 192, 256]), "chunk": rng.choice([32, 64, 100, 128, 256, 512]),
                "dtype": dtype, "qk": qk, "pv": pv}
    return {"kind": kind, "rows": _log(rng, 1, 12000), "cols": rng.choice([64, 128, 1000, 4096, 5120, 12288]),
            "dtype": rng.choice(["bfloat16", "float32", "float16"])}


# ---- inputs -------------------------------------------------------------------------------


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _rope(x: torch.Tensor, theta: float = 1.0e6) -> torch.Tensor:
    """Rotate-half RoPE over positions 0 .. L-1 in fp32."""
    length, dim = x.shape[-2:]
    inv = 1.0 / (theta ** (torch.arange(0, dim, 2, device=x.device, dtype=torch.float64) / dim))
    ang = torch.arange(length, device=x.device, dtype=torch.float64)[:, None] * inv[None, :]
    emb = torch.cat([ang, ang], dim=-1)
    half = torch.cat([-x[..., dim // 2:], x[..., :dim // 2]], dim=-1)
    return x * emb.cos().float() + half * emb.sin().float()


def _heads(gen, batch: int, heads: int, length: int, dim: int, dtype, rope: bool = False) -> torch.Tensor:
    """[B, H, L, D] activations: normalized heads with unequal channels, optionally rotated."""
    x = torch.randn((batch, heads, length, dim), device=DEVICE, generator=gen)
    x = x * torch.exp(0.4 * torch.randn((heads, 1, dim), device=DEVICE, generator=gen))
    return (_rope(x) if rope else x).to(dtype)


def _module(**kw) -> SimpleNamespace:
    """The attributes the attention reads from a transformer layer's attention module."""
    from faquant_amd.simulated_flash_attention import new_simulated_attention_stats

    attrs = dict(
        is_causal=True, training=False, faquant_attention_query_chunk_size=256,
        faquant_attention_key_chunk_size=128, faquant_qk_matmul_quant=True, faquant_pv_matmul_quant=True,
        faquant_pv_normalizer_mode="quantized_same", faquant_matmul_quant_kwargs=HIF4,
        faquant_simulated_attention_stats=new_simulated_attention_stats(),
    )
    attrs.update(kw)
    return SimpleNamespace(**attrs)


def _qkv(case: dict, seed: int):
    gen = _gen(seed)
    kind = case["kind"]
    if kind == "wan":  # [B, L, H, D], as Wan's modules hold them
        q, k, v = (_heads(gen, 1, case["heads"], n, 128, torch.bfloat16).transpose(1, 2).contiguous()
                   for n in (case["lq"], case["lk"], case["lk"]))
        return q, k, v
    if kind == "ablation":
        dtype = getattr(torch, case["dtype"])
        q = _heads(gen, 1, case["hq"], case["l"], case["d"], dtype, rope=True)
        k = _heads(gen, 1, case["hkv"], case["l"], case["d"], dtype, rope=True)
        return q, k, _heads(gen, 1, case["hkv"], case["l"], case["d"], dtype)
    lq = {"prefill": case.get("lq"), "padded": case.get("l"), "decode": 1}[kind]
    lk = case["lk"] if kind == "prefill" else case["l"]
    q = _heads(gen, case["batch"], case["hq"], lk if kind == "prefill" else lq, 128, torch.bfloat16,
               rope=True)[:, :, -lq:].contiguous()
    k = _heads(gen, case["batch"], case["hkv"], lk, 128, torch.bfloat16, rope=True)
    return q, k, _heads(gen, case["batch"], case["hkv"], lk, 128, torch.bfloat16)


def _padding(case: dict, seed: int) -> torch.Tensor:
    """[B, L] 0/1 mask of left-padded prompts: lengths from an eighth of L up, one of them L."""
    length = case["l"]
    g = torch.Generator().manual_seed(seed + 1)
    lens = torch.randint(max(1, length // 8), length + 1, (case["batch"],), generator=g)
    lens[0] = length
    return (torch.arange(length)[None, :] >= length - lens[:, None]).to(torch.int64).to(DEVICE)


def _linear_parts(case: dict, seed: int) -> SimpleNamespace:
    gen = _gen(seed)
    rows, k, n = case["rows"], case["k"], case["n"]
    # activations with a few large channels, weights of a trained layer's size
    x = torch.randn((rows, k), device=DEVICE, generator=gen)
    chan = torch.exp(0.5 * torch.randn((k,), device=DEVICE, generator=gen))
    parts = SimpleNamespace(x=(x * chan).to(torch.bfloat16))
    parts.w = (torch.randn((n, k), device=DEVICE, generator=gen) * 0.02).to(torch.bfloat16)
    parts.signs = parts.perm = parts.log = None
    if case["rotation"]:
        parts.signs = (torch.randint(0, 2, (k,), device=DEVICE, generator=gen) * 2 - 1).to(torch.int8)
        parts.perm = torch.randperm(k, device=DEVICE, generator=gen)
        parts.log = torch.rand((k,), device=DEVICE, generator=gen) - 0.5
    return parts


def _codec_input(case: dict, seed: int) -> torch.Tensor:
    gen = _gen(seed)
    x = torch.randn((case["rows"], case["cols"]), device=DEVICE, generator=gen) * 0.02
    x = x * torch.exp(0.5 * torch.randn((case["rows"], 1), device=DEVICE, generator=gen))
    return x.to(getattr(torch, case["dtype"]))


def prepare(case: dict, seed: int) -> SimpleNamespace:
    kind = case["kind"]
    st = SimpleNamespace(kind=kind)
    if kind == "codec":
        st.x = _codec_input(case, seed)
        return st
    if kind == "linear":
        from faquant_amd.quantization import FakeQuantLinear

        p = _linear_parts(case, seed)
        linear = torch.nn.Linear(case["k"], case["n"], bias=False, device="meta")
        linear.weight = torch.nn.Parameter(p.w, requires_grad=False)
        st.x = p.x
        st.layer = FakeQuantLinear(
            linear, quant_format="hif4", bits=4, weight_group_size=64, activation_group_size=64, symmetric=True,
            clip_ratio=1.0, input_rotation_signs=p.signs, input_rotation_permutation=p.perm,
            input_rotation_block_size=case["rotation"] or None,
            activation_min=-8.0 if p.log is not None else None, activation_max=8.0 if p.log is not None else None,
            activation_compand_log_scale=p.log, packed_weight=case["packed"]).to(DEVICE)
        return st
    st.q, st.k, st.v = _qkv(case, seed)
    if kind == "wan":
        from faquant_amd.wan22_attention import faquant_qdq, make_flash_attention

        st.attend = make_flash_attention(faquant_qdq(levels="123"), quantized_normalizer=True, qk_rotation=True)
        return st
    if kind == "prefill":
        st.module = _module(faquant_qk_rotation=True, faquant_qk_rotation_block_size=64)
    elif kind == "padded":
        st.module = _module()
        st.mask = _padding(case, seed)
    elif kind == "ablation":
        st.module = _module(faquant_attention_key_chunk_size=case["chunk"], faquant_qk_matmul_quant=case["qk"],
                            faquant_pv_matmul_quant=case["pv"])
    else:
        # the layer after the steps before: its caches hold the first l - 1 positions
        from faquant_amd.simulated_flash_attention import simulated_flash_attention_forward

        st.packed = case["packed"]
        st.module = _module(faquant_kv_cache_packed=st.packed)
        simulated_flash_attention_forward(st.module, st.q, st.k[:, :, :-1], st.v[:, :, :-1], None)
    return st


def _fork(module: SimpleNamespace) -> SimpleNamespace:
    """The module as it stood before the step, so that the step can be taken again (its dicts
    are copied, its cache buffers shared: a step writes the same new position into them)."""
    return SimpleNamespace(**{k: dict(v) if isinstance(v, dict) else v for k, v in vars(module).items()})


def run(state):
    kind = state.kind
    if kind == "codec":
        from faquant_amd.quantization import fake_quantize

        return fake_quantize(state.x, quant_format="hif4", bits=4, group_size=64)
    if kind == "linear":
        return state.layer(state.x)
    if kind == "wan":
        return state.attend(state.q, state.k, state.v)
    if kind == "prefill":
        from faquant_amd.qwen3 import attention_core

        return attention_core(state.module, state.q, state.k, state.v)
    from faquant_amd.simulated_flash_attention import simulated_flash_attention_forward

    if kind != "decode":
        return simulated_flash_attention_forward(state.module, state.q, state.k, state.v,
                                                 getattr(state, "mask", None))[0]
    module = _fork(state.module)
    out = simulated_flash_attention_forward(module, state.q, state.k, state.v, None)[0]
    caches = module.faquant_k_matmul_qdq_cache, module.faquant_v_matmul_qdq_cache
    if not state.packed:
        return [out, *caches]
    # the rows in use (a packed cache is allocated up to its capacity)
    return [out] + [t[:, :, :c.length] for c in caches for t in (c.codes, c.meta)]


# ---- work ---------------------------------------------------------------------------------


def _pairs(lq: int, lk: int, causal: bool) -> int:
    if not causal:
        return lq * lk
    return lq * (lk - lq) + lq * (lq + 1) // 2


def work(case: dict) -> dict:
    kind = case["kind"]
    size = {"bfloat16": 2, "float16": 2, "float32": 4}.get(case.get("dtype", "bfloat16"))
    if kind == "codec":
        n = case["rows"] * case["cols"]
        # group maximum, two exponents, scale, round, clamp and rescale of each value
        return {"bytes": 2 * size * n, "flops": 8.0 * n}
    if kind == "linear":
        rows, k, n = case["rows"], case["k"], case["n"]
        weight = n * k * 9 / 16 if case["packed"] else 2.0 * n * k
        return {"bytes": weight + 2.0 * rows * (k + n), "flops": 2.0 * rows * k * n}
    if kind == "decode":
        keys = case["batch"] * case["hkv"] * case["l"]
        # the caches of the earlier positions, the new position, the query and the output
        per_key = 144 if case["packed"] else 512
        return {"bytes": keys * per_key + 4.0 * case["batch"] * case["hq"] * 128,
                "flops": 4.0 * 128 * case["batch"] * case["hq"] * case["l"]}
    if kind == "wan":
        lq, lk, hq, hkv, batch, d, causal = case["lq"], case["lk"], case["heads"], case["heads"], 1, 128, False
    elif kind == "prefill":
        lq, lk, hq, hkv, batch, d, causal = case["lq"], case["lk"], case["hq"], case["hkv"], case["batch"], 128, True
    else:
        lq = lk = case["l"]
        hq, hkv, batch, d, causal = case["hq"], case["hkv"], case.get("batch", 1), case.get("d", 128), True
    pairs = _pairs(lq, lk, causal)
    if kind == "padded":
        pairs *= 0.42  # prompt lengths between an eighth and the whole: the mean of their squares
    return {"bytes": size * batch * d * (2.0 * hq * lq + 2.0 * hkv * lk), "flops": 4.0 * d * batch * hq * pairs}


# ---- float64 -------------------------------------------------------------------------------


def _bf16(x: torch.Tensor) -> torch.Tensor:
    """float64 rounded to bf16 through fp32 (the format's own definition), back in float64."""
    return x.float().to(torch.bfloat16).double()


def _pow2_floor(x: torch.Tensor) -> torch.Tensor:
    return torch.exp2(torch.floor(torch.log2(x)))


def _hif4(x: torch.Tensor) -> torch.Tensor:
    """HiF4 (levels 123) quantize-dequantize of float64 x along its last axis in 64-value groups."""
    size = x.shape[-1]
    pad = -size % 64
    if pad:
        x = torch.nn.functional.pad(x, (0, pad))
    g = x.reshape(*x.shape[:-1], -1, 8, 2, 4)
    mag = g.abs()
    m3 = mag.amax(-1, keepdim=True)
    m2 = m3.amax(-2, keepdim=True)
    s = _bf16(m2.amax(-3, keepdim=True) * 0.142578125).clamp(2.0**-48, 49152.0)
    step = _pow2_floor(s) / 4
    s = torch.round(s / step) * step  # two significand bits, ties to even
    rec = _bf16(1.0 / s)
    k2 = (m2 * rec >= 4).double()
    k3 = (m3 * rec >= 2 * torch.exp2(k2)).double()
    mult = torch.exp2(k2 + k3)
    code = torch.floor(mag * rec / mult * 4 + 0.5).clamp_(max=7)
    y = torch.sign(g) * code * (mult * s / 4)
    return y.reshape(x.shape)[..., :size]


def _exact_attention(q, k, v, *, chunk: int, quant_p: bool, causal: bool, valid=None) -> torch.Tensor:
    """Tiled attention in float64 of [B, H, L, D] operands (already quantized); [B, Lq, Hq, D].
    P is taken against the running maximum after each key tile, as the tiled recurrence does."""
    batch, hq, lq, d = q.shape
    hkv, lk = k.shape[1:3]
    out = torch.empty((batch, lq, hq, d), device=q.device, dtype=torch.float64)
    rows = max(16, min(lq, (1 << 25) // max(lk, 1)))
    for b in range(batch):
        for h in range(hq):
            kh, vh = k[b, h * hkv // hq].double(), v[b, h * hkv // hq].double()
            for r0 in range(0, lq, rows):
                r1 = min(lq, r0 + rows)
                end = min(lk, r1 + lk - lq) if causal else lk
                tiles = -(-end // chunk)
                s = q[b, h, r0:r1].double() @ kh[:end].T * d**-0.5
                if causal:
                    pos = torch.arange(r0, r1, device=q.device)[:, None] + (lk - lq)
                    s.masked_fill_(torch.arange(end, device=q.device)[None, :] > pos, -math.inf)
                if valid is not None:
                    s.masked_fill_(~valid[b, None, :end], -math.inf)
                s = torch.nn.functional.pad(s, (0, tiles * chunk - end), value=-math.inf).view(r1 - r0, tiles, chunk)
                m = s.amax(-1).cummax(1).values
                top = m[:, -1:]
                p = torch.exp(s - torch.where(torch.isinf(m), torch.zeros_like(m), m)[..., None])
                del s
                ph = _hif4(p) if quant_p else p
                ph = ph * torch.exp(m - torch.where(torch.isinf(top), torch.zeros_like(top), top))[..., None]
                ph = ph.view(r1 - r0, -1)[:, :end]
                den = ph.sum(-1, keepdim=True)
                o = torch.where(den > 0, ph @ vh[:end] / den.clamp(min=1e-300), torch.zeros_like(den))
                if valid is not None:
                    o = o * valid[b, r0 + lk - lq:r1 + lk - lq, None]
                out[b, r0:r1, h] = o
    return out


def _rotate(x: torch.Tensor, block: int) -> torch.Tensor:
    """Normalized Walsh-Hadamard transform of each block along the last axis, in float64."""
    shape = x.shape
    y = x.double().reshape(-1, block)
    step = 1
    while step < block:
        y = y.view(-1, block // (2 * step), 2, step)
        y = torch.stack((y[:, :, 0] + y[:, :, 1], y[:, :, 0] - y[:, :, 1]), 2).view(-1, block)
        step *= 2
    return (y / math.sqrt(block)).view(shape)


def _exact_linear(case: dict, seed: int) -> torch.Tensor:
    p = _linear_parts(case, seed)
    w = torch.cat([_hif4(rows.double()) for rows in p.w.split(1024)])
    scale = None if p.log is None else _bf16(p.log.double().exp())
    out = []
    for rows in p.x.split(512):
        x = rows.double()
        if p.signs is not None:
            x = _bf16(_rotate((x * p.signs.double())[:, p.perm], case["rotation"]))
            x = _bf16(x.clamp(-8.0, 8.0) * scale)
        x = _hif4(x)
        if scale is not None:
            x = _bf16(x / scale)
        out.append(x @ w.T)
    return torch.cat(out)


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "codec":
        x = _codec_input(case, seed)
        return torch.cat([_hif4(rows.double()) for rows in x.split(1024)])
    if kind == "linear":
        return _exact_linear(case, seed)
    q, k, v = _qkv(case, seed)
    if kind == "wan":
        q, k, v = (t.transpose(1, 2) for t in (q, k, v))
        q, k = _bf16(_rotate(q, 128)), _bf16(_rotate(k, 128))
    elif kind == "prefill":
        q, k = _bf16(_rotate(q, 64)), _bf16(_rotate(k, 64))
    qk, pv = case.get("qk", True), case.get("pv", True)
    small = torch.float16 if case.get("dtype") == "float16" else None  # a quantized operand keeps its dtype

    def operand(t, quantize):
        if not quantize:
            return t
        y = torch.cat([_hif4(h.double()) for h in t.split(1, dim=1)], dim=1)
        return y.float().to(small).double() if small else y

    valid = None
    if kind == "padded":
        valid = _padding(case, seed).bool()
    k, v = operand(k, qk), operand(v, pv)
    out = _exact_attention(operand(q, qk), k, v, chunk=case.get("chunk", 128), quant_p=pv, causal=kind != "wan",
                           valid=valid)
    if kind == "decode":  # and the caches after the step; their packed words are no numbers
        return [out, None, None, None, None] if case["packed"] else [out, k, v]
    return out


def tolerance(case: dict):
    kind = case["kind"]
    if kind == "codec":
        return "exact"  # the codes are integers and their scales a format's numbers
    if kind == "linear":
        return {"rel": 8e-3}  # bf16 results of bf16 operands
    if case.get("dtype") == "float32":
        # a P code on a boundary moves with the last bit of a score; without P codes fp32 sums
        return {"rel": 2e-3 if case["pv"] else 1e-5}
    if case.get("dtype") == "float16":
        return {"rel": 2e-3}
    return {"rel": 8e-3}  # bf16 outputs
