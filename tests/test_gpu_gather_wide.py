"""The plain delivery with 128 features per workgroup (BF16, FP8) against the
oracle's gather: every alignment class of its LDS reads, patches with and
without a padded last k-step, ragged position tiles, accumulate, and the
geometries beside it that keep 64 features (short patches, too few workgroups,
an odd number of rounds of them, features not a multiple of 128).
Operands are small integers times powers of two, exact in both formats, whose
products and sums are exact in FP32 too: the results are equal."""
import numpy as np
import pytest
import torch

import oracle as O
from openpv_amd import abi, runtime as R

pytestmark = pytest.mark.gpu

CASES = [
    # source (nbatch, nx, ny, nf, halo), target, post-perspective patch
    ((16, 64, 64, 8, 4), (16, 32, 32, 256, 0), 8),    # 8-aligned, several k groups
    ((32, 40, 72, 4, 2), (32, 20, 36, 256, 0), 4),    # ragged tiles, K 64
    ((32, 64, 64, 2, 4), (32, 16, 16, 512, 0), 12),   # stride 4: K 288, 9 k-steps
    ((64, 36, 36, 2, 2), (64, 18, 18, 128, 0), 4),    # 4-aligned, one k-step
    ((64, 34, 34, 3, 4), (64, 17, 17, 128, 0), 8),    # 2-aligned, rows of 24 values
    ((1, 32, 32, 8, 4), (1, 16, 16, 256, 0), 8),      # too few workgroups
    ((16, 64, 64, 8, 4), (16, 32, 32, 192, 0), 8),    # not a multiple of 128
    ((16, 64, 64, 8, 4), (16, 32, 32, 256, 0), 10),   # 8-aligned, K 800: BF16 takes 128
    ((16, 64, 64, 12, 4), (16, 32, 32, 256, 0), 10),  # ... K 1200: half of the last k-step is padding
    ((2, 32, 32, 4, 2), (2, 16, 16, 128, 0), 6),      # 64 features, K 144: a padded last k-step
    ((64, 64, 64, 3, 6), (64, 16, 16, 256, 0), 16),   # 4-aligned, K 768, stride 4: BF16 takes 128
    ((40, 36, 34, 1, 12), (40, 18, 17, 256, 0), 24),  # 2-aligned, K 576, ragged: both take 128, 480 workgroups
    ((24, 64, 64, 5, 4), (24, 32, 32, 256, 0), 8),    # 2-aligned, K 320, 384 workgroups: both take 128
    ((17, 36, 36, 16, 2), (17, 18, 18, 384, 0), 6),   # starts 32 values apart, K 576, 306 workgroups: 64
    ((64, 32, 32, 16, 2), (64, 16, 16, 256, 0), 6),   # ... with 256: BF16 takes 128
    ((64, 36, 36, 1, 4), (64, 18, 18, 128, 0), 8),    # 2-aligned, K 64, 384 workgroups: 64
    ((64, 32, 32, 1, 4), (64, 16, 16, 256, 0), 8),    # ... with 256: FP8 takes 128
]


@pytest.mark.parametrize("arith", [abi.ARITH_BF16, abi.ARITH_FP8])
@pytest.mark.parametrize("case", CASES)
def test_wide_gather_exact_on_representable_values(case, arith):
    st, tt, p = case
    rng = np.random.default_rng(17)
    hs, os_ = abi.Loc.make(*st[:4], halo=st[4]), O.Loc.make(*st[:4], halo=st[4])
    ht, ot = abi.Loc.make(*tt[:4], halo=tt[4]), O.Loc.make(*tt[:4], halo=tt[4])
    W = rng.integers(-4, 5, (ht.nf, p, p, hs.nf)).astype(np.float32) / 8
    W[:, 0, 0, 0] = 0.5                              # every kernel has the same FP8 scale
    A = rng.integers(-6, 7, hs.nbatch * hs.num_ext).astype(np.float32) / 4
    d = R.PostsynapticPerspectiveGPUDelivery(hs, ht, p, p, torch.as_tensor(W.ravel()).cuda(), arith=arith)
    d.set_source_scale(16.0)
    ref = O.recv_post(os_, ot, p, p, A, W)
    for accumulate in (False, True):
        g = torch.full((ht.nbatch * ht.num_res,), 3.0, device="cuda")
        d.deliver(torch.as_tensor(A).cuda(), g, accumulate=accumulate)
        torch.cuda.synchronize()
        assert np.array_equal(g.cpu().numpy(), ref + (3.0 if accumulate else 0.0))
