"""hk_unified_reduce_sum_f32 over an outer axis: columns that end inside a group of four or of 256,
rows that end inside a round of eight or a slice, rows and inputs at odd offsets, several runs of
columns (runs of a multiple of four take 16-byte loads, others single ones). Small whole numbers,
so every order of adding them is exact and the sums have to be equal; NaN around what is read."""
from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("length", [1, 3, 29, 32, 33, 64, 131, 4099])
@pytest.mark.parametrize("runs,inner,pad,off", [(1, 3, 0, 0), (1, 4, 0, 0), (1, 5, 2, 1),
                                                (1, 255, 0, 3), (1, 257, 1, 0), (1, 1024, 4, 2),
                                                (5, 4, 3, 1), (3, 260, 0, 0), (6, 33, 0, 0)])
def test_outer_sums_are_exact(hk, runs, inner, pad, off, length):
    print("[case] reduce outer", runs, inner, pad, off, length, flush=True)
    g = np.random.default_rng(inner * 31 + length)
    row = inner + pad
    x = g.integers(-9, 10, (runs, length, inner)).astype(np.float32)
    buf = np.full((runs, length, row), np.nan, np.float32)
    buf[:, :, :inner] = x
    src = torch.full((off + buf.size + 8,), float("nan"), device="cuda")
    src[off:off + buf.size] = torch.from_numpy(buf.reshape(-1)).cuda()
    nout = runs * inner
    layout = hk.ReductionLayout(hk.REDUCE_OUTER, nout, length, length * row, inner, row)
    want = x.astype(np.float64).sum(1).reshape(-1)
    got = hk.unified_reduce_sum(src[off:], layout).cpu().numpy()
    assert np.array_equal(got, want)


@pytest.mark.parametrize("nout,inner", [(10, 8), (21, 8), (262, 256), (7, 4), (12, 8), (9, 16)])
def test_outputs_end_inside_a_run(hk, nout, inner):
    # num_outputs is no whole number of runs: the last outputs are the first columns of the last run
    length, runs = 37, -(-nout // inner)
    print("[case] reduce outer part run", nout, inner, flush=True)
    x = np.random.default_rng(nout).integers(-9, 10, (runs, length, inner)).astype(np.float32)
    layout = hk.ReductionLayout(hk.REDUCE_OUTER, nout, length, length * inner, inner, inner)
    want = x.astype(np.float64).sum(1).reshape(-1)[:nout]
    got = hk.unified_reduce_sum(torch.from_numpy(x).cuda(), layout).cpu().numpy()
    assert np.array_equal(got, want)
