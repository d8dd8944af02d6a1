"""The FP32 channel GEMM's default number of channel ranges where the caller's
scratch holds fewer partials than it takes (sized for another batch): it
halves until they fit, with the bits of that number given explicitly; an
explicit number without room, and no scratch at all, run as one range."""
import numpy as np
import pytest
import torch

from openpv_amd import abi, runtime as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("held,ranges", [(4, 4), (3, 2), (2, 2), (1, 1), (0, 1)])
def test_default_ranges_follow_the_scratch(held, ranges):
    rng = np.random.default_rng(12)
    src, tgt, p = abi.Loc.make(3, 16, 12, 128, 2), abi.Loc.make(3, 32, 24, 3, 0), 4   # post patch of an 8x8 one
    W = torch.as_tensor(rng.standard_normal(4 * 3 * p * p * 128).astype(np.float32) * 0.05).cuda()
    A = torch.as_tensor(rng.standard_normal(src.nbatch * src.num_ext).astype(np.float32)).cuda()
    n = tgt.nbatch * tgt.num_res

    def deliver(splits, floats):
        d = R.PostsynapticPerspectiveGPUDelivery(src, tgt, p, p, W, arith=abi.ARITH_FP32, split=False)
        d.cgemm_splits = splits
        d.scratch = torch.empty(floats, device="cuda") if floats else None
        g = torch.empty(n, device="cuda")
        d.deliver(A, g, accumulate=False)
        torch.cuda.synchronize()
        return g.view(torch.int32)

    by_number = {k: deliver(k, k * n) for k in (1, 2, 4)}
    assert not torch.equal(by_number[1], by_number[2]) and not torch.equal(by_number[2], by_number[4])
    assert torch.equal(deliver(0, held * n), by_number[ranges])
    if held < 4:
        assert torch.equal(deliver(4, held * n), by_number[1])
