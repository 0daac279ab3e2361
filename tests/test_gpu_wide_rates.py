"""K = 5 .. 8 (n = 80, 96, 112, 128) on the GEMV's lane reader, dense and routed, against the oracle."""
import numpy as np
import pytest
import torch

import oracle as O
from sushi_amd import exl3, synth
from tests._util import max_abs_rel
from tests.test_gpu_moe import BAR, _np, _route, _to
from tests.test_gpu_parity import DECODES, Dense, _hold

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("label", ["mcg", "3inst", "mul1", "spec1"])
@pytest.mark.parametrize("n,rows", [(80, 1), (80, 5), (96, 2), (96, 16), (112, 1), (112, 7), (128, 1), (128, 9)])
def test_gemv_wide_rates(dev, label, n, rows):
    """Every template of the reader's rates, on k spans of an odd number of 128-blocks (384: one, three and more tiles
    a wave), held to the summand bar with its window and flipped-bit mutations."""
    d = Dense(dev, 900 + n + rows, rows, 384, 256, n)
    dec, odec = DECODES[label]
    _hold(d.inner(dec), d, odec, seed=n + rows, what=f"wide {label} n={n} rows={rows}")


@pytest.mark.parametrize("n,rows", [(80, 2), (96, 12), (112, 3), (128, 20)])
def test_moe_wide_rates(dev, n, rows):
    """The routed chain at those rates: per slot (up to 8 rows) and in expert windows, with a fused shared bank."""
    E, hidden, inter, k = 8, 256, 384, 2
    b, sh = (synth.bank(91, nm, e, hidden, inter, n, norm=True) for nm, e in (("wide", E), ("wide.shared", 1)))
    x = synth.normal(91, f"x{rows}", (rows, hidden))
    inds, scores = _route(91 + rows, rows, E, k)
    args = (hidden, inter, (n, n, n), O.decode(O.CB_MCG))
    routed = O.moe_swiglu_rows(x.float().numpy(), _np(b.gate), _np(b.up), _np(b.down), inds, scores, *args, threads=8)
    shared = O.moe_swiglu_rows(x.float().numpy(), _np(sh.gate), _np(sh.up), _np(sh.down), np.zeros((rows, 1)),
                               np.ones((rows, 1)), *args, threads=8)
    want = routed.astype(np.float16).astype(np.float32) + shared.astype(np.float16).astype(np.float32)
    y = exl3.moe_with_shared_bank(x.to(dev), _to(b, dev), _to(sh, dev), torch.from_numpy(inds.view(np.int32)).to(dev),
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
