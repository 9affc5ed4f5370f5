"""The allocation-free solve of batches whose fastest layouts need more scratch
than there is: served in layouts that fit, the same scores as the allocating
entry's, a sample against the oracle."""

import numpy as np
import pytest
import torch

import oracle as O
import pyalign_amd as pa
from pyalign_amd import algorithm
from tests.test_gpu_band import LOCS
from tests.test_zz_no_alloc import _both, _same, _solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,most_s,most_t,loc,form", [(276247, 67, 531, "global", "indexed"),
                                                      (255324, 73, 355, "global", "binary"),
                                                      (318456, 44, 431, "local", "binary")])
def test_fits(n, most_s, most_t, loc, form):
    k = np.arange(n, dtype=np.uint64)
    ls = (1 + (k * 2654435761 % 2**32 >> 8) % most_s).astype(np.int32)
    lt = (1 + (k * 40503 % 2**32 >> 4) % most_t).astype(np.int32)
    rng = np.random.default_rng(n)
    codes = rng.integers(0, 4, 5000).astype(np.uint8 if form == "indexed" else np.int32)
    off_s, off_t = (rng.integers(0, 4400, n) for _ in range(2))  # (all within the same codes)
    table = np.where(np.eye(4), 2, -1).astype(np.float32)
    dev = torch.from_numpy(codes).cuda()
    extra = dict(table=table) if form == "indexed" else dict(eq=2.0, ne=-1.0)
    rg, keep = algorithm.make_ragged(form, ls, lt, codes_s=dev.data_ptr(), codes_t=dev.data_ptr(), off_s=off_s,
                                     off_t=off_t, on_device=True, **extra)
    torch.cuda.synchronize()
    ref, got = _both(_solver(LOCS[loc][0], pa.AffineGapCost(2, 0.5), 512, 1024), rg, n)
    del keep
    assert not np.isnan(got).any() and _same(ref, got)
    for q in range(0, n, n // 40):
        S = table[codes[off_s[q]:off_s[q] + ls[q]]][:, codes[off_t[q]:off_t[q] + lt[q]]]
        want = O.OracleResult(O.make_config(locality=LOCS[loc][1], gap=("affine", 2, 0.5), goal=O.GOAL_SCORE, lim_s=512,
                                            lim_t=1024), S)
        assert got[q].tobytes() == want.score.tobytes(), q
