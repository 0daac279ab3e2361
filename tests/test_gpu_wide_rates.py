"""K = 5 .. 8 (n = 80, 96, 112, 128) on the lane readers of the GEMV, dense and routed, and of the dense GEMM, against the
oracle."""
import numpy as np
import pytest
import torch

import oracle as O
from sushi_amd import exl3, synth
from tests import _parity as P
from tests._util import max_abs_rel
from tests.test_gpu_moe import BAR, _np, _route, _to
from tests.test_gpu_parity import DECODES, Dense, _hold, _u16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("label", ["mcg", "3inst", "mul1", "spec1"])
@pytest.mark.parametrize("n,rows", [(80, 1), (80, 5), (96, 2), (96, 16), (112, 1), (112, 7), (128, 1), (128, 9)])
def test_gemv_wide_rates(dev, label, n, rows):
    """Every template of the reader's rates, over three 128-blocks of k in three splits (one k-tile a wave), held to the
    summand bar with its window and flipped-bit mutations."""
    d = Dense(dev, 900 + n + rows, rows, 384, 256, n)
    dec, odec = DECODES[label]
    _hold(d.inner(dec), d, odec, seed=n + rows, what=f"wide {label} n={n} rows={rows}")


@pytest.mark.parametrize("in_f", [384, 640, 1024])
@pytest.mark.parametrize("rows", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("n", [80, 96, 112, 128])
def test_gemv_wide_rates_several_tiles_a_wave(dev, n, rows, in_f):
    """One split, so a wave runs 3, 5 or 8 k-tiles: the second tile in flight, the refill of a decoded slot's words and
    the tail behind it, at every row template (the rows kept whole), the codebooks in turn."""
    d = Dense(dev, 930 + n + rows, rows, in_f, 256, n)
    label = ("mcg", "3inst", "mul1", "spec1")[(n // 16 + rows.bit_length() + in_f // 128) % 4]
    dec, odec = DECODES[label]
    with exl3.arm_overrides(gemv_splits=1, gemv_rows_per_group=16):
        got = d.inner(dec)
    _hold(got, d, odec, seed=n + rows, what=f"wide {label} n={n} rows={rows} in={in_f}")


@pytest.mark.parametrize("splits", [0, 1])
@pytest.mark.parametrize("n,rows", [(80, 2), (96, 12), (112, 3), (128, 20)])
def test_moe_wide_rates(dev, n, rows, splits):
    """The routed chain at those rates, per slot (up to 8 rows) and in expert windows, with a shared bank: the default
    splits (one k-tile a wave here) and one split (two for gate and up, three for down)."""
    E, hidden, inter, k = 8, 256, 384, 2
    b, sh = (synth.bank(91, nm, e, hidden, inter, n, norm=True) for nm, e in (("wide", E), ("wide.shared", 1)))
    x = synth.normal(91, f"x{rows}", (rows, hidden))
    inds, scores = _route(91 + rows, rows, E, k)
    args = (hidden, inter, (n, n, n), O.decode(O.CB_MCG))
    routed = O.moe_swiglu_rows(x.float().numpy(), _np(b.gate), _np(b.up), _np(b.down), inds, scores, *args, threads=8)
    shared = O.moe_swiglu_rows(x.float().numpy(), _np(sh.gate), _np(sh.up), _np(sh.down), np.zeros((rows, 1)),
                               np.ones((rows, 1)), *args, threads=8)
    want = routed.astype(np.float16).astype(np.float32) + shared.astype(np.float16).astype(np.float32)
    with exl3.arm_overrides(**(dict(moe_splits1=splits, moe_splits2=splits) if splits else {})):
        y = exl3.moe_with_shared_bank(x.to(dev), _to(b, dev), _to(sh, dev),
                                      torch.from_numpy(inds.view(np.int32)).to(dev),
                                      torch.from_numpy(scores).to(dev), exl3.MCG)
    assert max_abs_rel(y.float().cpu().numpy(), want) < BAR


@pytest.mark.parametrize("label", ["mcg", "3inst", "mul1", "spec1"])
@pytest.mark.parametrize("n,rows", [(80, 17), (80, 300), (96, 40), (96, 257), (112, 130), (112, 16 * 8 + 1), (128, 64),
                                    (128, 520)])
def test_gemm_wide_rates(dev, label, n, rows):
    """The GEMM tile at those rates: one to three row tiles with tails, four and eight decode waves (the switch lies at
    128 rows), k of three 128-blocks, held as the GEMV is."""
    d = Dense(dev, 940 + n + rows, rows, 384, 256, n)
    dec, odec = DECODES[label]
    _hold(d.inner(dec), d, odec, seed=n + rows, what=f"wide gemm {label} n={n} rows={rows}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,rows,label", [(80, 40, "spec1"), (96, 200, "mcg"), (112, 17, "mul1"), (128, 300, "3inst")])
def test_gemm_wide_rates_activation_dtypes(dev, n, rows, label, dtype):
    """bf16 and f32 inputs (rounded to f16 as prepareInput does), the f32 output to the summand bar; the 16-bit output
    is that output rounded once."""
    d = Dense(dev, 960 + n, rows, 384, 256, n)
    x = d.xd.to(dtype)
    d.p = P.prepared_rows(x.float().cpu().numpy(), d.suh)
    dec, odec = DECODES[label]
    y = exl3.linear(x, d.pd, dec, out_dtype=torch.float32)
    _hold(P.inner_from_output(y.cpu().numpy(), d.svh), d, odec, seed=n, what=f"wide gemm {label} n={n} {dtype}")
    assert torch.equal(exl3.linear(x, d.pd, dec), y.to(dtype))


@pytest.mark.parametrize("n,rows,label", [(80, 17, "mcg"), (96, 40, "3inst"), (112, 130, "spec1"), (128, 257, "mul1")])
def test_gemm_wide_rates_grouped(dev, n, rows, label):
    """Three weight groups in one call, each held to the summand bar."""
    groups, in_f, out_f = 3, 384, 256
    p = synth.proj(970 + n, "wideg", groups, in_f, out_f, n)
    x = synth.normal(970 + n, "wideg.x", (groups, rows, in_f))
    dec, odec = DECODES[label]
    pd = exl3.Proj(p.trellis.to(dev), p.suh.to(dev), p.svh.to(dev))
    y = exl3.linear_grouped(x.float().to(dev), pd, dec).cpu().numpy()  # f32 x: f32 outputs
    for g in range(groups):
        t = P.truth(P.prepared_rows(x[g].float().numpy(), _u16(p.suh)[g]),
                    P.decoded(_u16(p.trellis)[g], in_f, out_f, n, odec))
        why = P.verdict(P.inner_from_output(y[g], _u16(p.svh)[g]), t)
        assert why is None, f"{label} n={n} group {g}: {why}"
