"""Activation counts of the MFMA Hebbian forms (whole windows counted while the
activity is staged, cut ones by the border kernel, prefix sums in the reduce)
against the oracle, exactly: layers without a whole window along one or both
axes, ragged features, several item blocks, runs longer than one segment,
every split of the rows, and counts accumulated over two calls."""
import numpy as np
import pytest
import torch

import oracle as O
from openpv_amd import abi, runtime as R

pytestmark = pytest.mark.gpu
DEV = "cuda"

CASES = [
    # pre (nbatch, nx, ny, nf, halo), post, patch, rows per chunk (0: the default)
    ((1, 3, 3, 70, 2), (1, 12, 12, 1, 6), 16, 0),      # no whole window
    ((2, 40, 3, 65, 2), (2, 160, 12, 1, 6), 16, 1),    # whole along x only; a run of 32 and a rest
    ((1, 4, 37, 8, 1), (1, 8, 74, 3, 2), 6, 5),        # ... along y only
    ((2, 12, 10, 130, 2), (2, 24, 20, 3, 3), 8, 0),    # two feature blocks and a ragged one
    ((1, 9, 9, 40, 2), (1, 36, 36, 2, 6), 16, 3),      # two item blocks
    ((1, 140, 6, 16, 1), (1, 280, 12, 1, 1), 4, 0),    # several 32-column steps a row
    ((3, 6, 6, 20, 1), (3, 6, 6, 2, 1), 3, 7),         # one to one
    # post rows longer than the 768 elements whose loads are issued a row ahead,
    # windows of over 80 KB (a ring of nyp rows, two barriers a row), chunks that
    # walk several pre rows and cross from one image to the next
    ((2, 64, 4, 20, 2), (2, 256, 16, 3, 6), 16, 5),
    ((2, 20, 5, 16, 1), (2, 160, 40, 3, 8), 24, 100),  # eight new post rows a pre row
    # eight new post rows where the ring has room for them, and fewer than 256 elements each
    ((2, 5, 7, 70, 1), (2, 40, 56, 1, 4), 16, 6),
]


@pytest.mark.parametrize("arith", [abi.ARITH_FP32, abi.ARITH_BF16])
@pytest.mark.parametrize("case", CASES)
def test_hebbian_counts_equal_oracle(case, arith):
    pt, qt, p, rows = case
    rng = np.random.default_rng(91)
    hp, op = abi.Loc.make(*pt[:4], halo=pt[4]), O.Loc.make(*pt[:4], halo=pt[4])
    hq, oq = abi.Loc.make(*qt[:4], halo=qt[4]), O.Loc.make(*qt[:4], halo=qt[4])
    a = rng.standard_normal(hp.nbatch * hp.num_ext).astype(np.float32)
    a[rng.random(a.shape) < 0.6] = 0                    # the halo's neurons are active too
    a[a > 2.0] *= np.float32(1e-41)                     # active, below the normal range
    r = rng.standard_normal(hq.nbatch * hq.num_ext).astype(np.float32)
    dw, cnt = O.hebbian_dw(op, oq, p, p, oq.nf, 0.25, a, r, counts=True)
    hb = R.HebbianUpdater(hp, hq, p, p, 0.25, normalize_dw=True, device=DEV)
    hb.rows_per_chunk = rows
    da, dr = torch.as_tensor(a).to(DEV), torch.as_tensor(r).to(DEV)
    hb.update_dw(da, dr, arith=arith)
    torch.cuda.synchronize()
    assert np.array_equal(hb.counts.cpu().numpy(), cnt)
    err = np.abs(hb.dw.cpu().numpy() - dw)
    if arith == abi.ARITH_FP32:                         # FP32 products, another order of the sums
        assert err.max() <= 2e-5 * np.abs(dw).max()
    else:                                               # operands rounded to 8 bits
        assert np.sqrt((err ** 2).mean()) <= 1e-2 * np.sqrt((dw ** 2).mean())
    hb.update_dw(da, dr, clear=False, arith=arith)
    torch.cuda.synchronize()
    assert np.array_equal(hb.counts.cpu().numpy(), 2 * cnt)
