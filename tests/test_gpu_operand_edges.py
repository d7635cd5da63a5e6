"""The operand prologue's quantizer (natural rows and V^T) against the oracle, bit for bit, on groups
where its short forms could go wrong: signed zeros, subnormals, the scale clamps, values on
code boundaries and micro-exponent thresholds, infinities and NaN groups, every level form."""

from __future__ import annotations

import numpy as np
import pytest

from oracle import hif4 as OQ

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _rows():
    g = np.random.default_rng(7)
    x = g.standard_normal((40, 128)).astype(np.float32)
    x[0] = 0.0
    x[1, ::2] = -0.0
    x[2] *= np.float32(1e-40)  # subnormal
    x[3] *= np.float32(2.0**-52)  # below the smallest scale
    x[4] *= np.float32(1e38)  # above the largest
    x[5, 3], x[5, 70] = np.inf, -np.inf
    x[6, 10] = np.nan  # one NaN group, one plain
    x[7, 64:] = np.nan
    x[8] = np.where(np.arange(128) % 2, 1.75, -1.75)
    for r in range(9, 40):  # multiples of a quarter around every threshold of a power-of-two scale
        s = np.float32(2.0 ** (r - 24))
        x[r] = s * (g.integers(-29, 30, 128) / np.float32(4.0) + g.choice([0, 2.0**-9, -(2.0**-9)], 128))
        x[r, ::64] = 7 * s
    return x.astype(np.float32)


@pytest.mark.parametrize("levels", ["123", "12", "13"])
@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_operand_quantizer_edges(dev, levels, dtype):
    from faquant_amd import _ops

    x = _rows()
    if dtype == "bfloat16":
        x = OQ.bf16_round(x)
    with np.errstate(invalid="ignore", over="ignore"):
        want = OQ.fake_quantize_hif4(x, levels, dtype=dtype)
    t = torch.from_numpy(x).to(dev, getattr(torch, dtype))[None, None]
    rows = _ops.operand_prep(t, levels=levels)[0][0, 0].float().cpu().numpy()
    vt = _ops.operand_prep_vt(t, levels=levels)[0, 0, :, :40].T.float().cpu().numpy()
    act = _ops.act_qdq_rows(t[0, 0].contiguous(), levels=levels).float().cpu().numpy()
    nan = np.isnan(want)
    for got in (rows, vt, act):
        assert np.array_equal(np.isnan(got), nan)
        assert np.array_equal(got[~nan].view(np.uint32), want[~nan].view(np.uint32))


@pytest.mark.parametrize("bounds", [(float("nan"), 1.0), (-1.0, float("nan")), (float("nan"), float("nan"))])
def test_a_nan_clamp_bound_bounds_nothing(dev, bounds):
    from faquant_amd import _ops

    x = torch.randn((5, 256), generator=torch.Generator().manual_seed(3)).to(dev, torch.bfloat16)
    lo, hi = bounds
    want = _ops.act_prep_rows(x, levels="123", act_min=None if lo != lo else lo, act_max=None if hi != hi else hi)
    assert torch.equal(_ops.act_prep_rows(x, levels="123", act_min=lo, act_max=hi), want)
