"""The vector-ALU gather with 64 features per workgroup, which needs more than 32
features and at least 256 workgroups (fewer take 32 features each), against
the oracle: ragged position tiles, a ragged last feature block, accumulate, and
the layer update in the epilogue.  EXACT bit for bit; FP32 (patches of a size
that is no multiple of 32, which the matrix cores do not take) within 1e-5 of
the largest value."""
import numpy as np
import pytest
import torch

import oracle as O
from openpv_amd import abi, runtime as R

pytestmark = pytest.mark.gpu
FMAX = float(np.finfo(np.float32).max)

CASES = [
    # source (nbatch, nx, ny, nf, halo), target, post-perspective patch; workgroups
    ((22, 40, 22, 3, 3), (22, 20, 11, 70, 1), 6),     # 22 x 3 x 2 tiles x 2 blocks = 264
    ((32, 64, 64, 1, 6), (32, 16, 16, 96, 2), 12),    # 256, stride 4
    ((37, 9, 17, 5, 2), (37, 9, 17, 104, 0), 5),      # one to one; 444
]


@pytest.mark.parametrize("arith", [abi.ARITH_EXACT, abi.ARITH_FP32])
@pytest.mark.parametrize("case", CASES)
def test_tiled_gather(case, arith):
    st, tt, p = case
    rng = np.random.default_rng(53)
    hs, os_ = abi.Loc.make(*st[:4], halo=st[4]), O.Loc.make(*st[:4], halo=st[4])
    ht, ot = abi.Loc.make(*tt[:4], halo=tt[4]), O.Loc.make(*tt[:4], halo=tt[4])
    assert (p * p * hs.nf) % 32
    assert -(-ht.nx // 8) * -(-ht.ny // 8) * -(-ht.nf // 64) * ht.nbatch >= 256
    W = (rng.standard_normal((ht.nf, p, p, hs.nf)) * 0.05).astype(np.float32)
    A = rng.standard_normal(hs.nbatch * hs.num_ext).astype(np.float32)
    n = ht.nbatch * ht.num_res
    base = rng.standard_normal(n).astype(np.float32)
    dA = torch.as_tensor(A).cuda()
    d = R.PostsynapticPerspectiveGPUDelivery(hs, ht, p, p, torch.as_tensor(W.ravel()).cuda(), arith=arith)
    for accumulate in (False, True):
        ref = O.recv_post(os_, ot, p, p, A, W, gsyn=base.copy() if accumulate else None)
        g = torch.as_tensor(base).cuda()
        d.deliver(dA, g, accumulate=accumulate)
        torch.cuda.synchronize()
        got = g.cpu().numpy()
        if arith == abi.ARITH_EXACT:
            assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))
        else:
            assert np.abs(got - ref).max() <= 1e-5 * np.abs(ref).max()
    # the update in the epilogue: the delivery followed by the layer's own update
    g = torch.zeros(n, device="cuda")
    d.deliver(dA, g, accumulate=False)
    for vertices in (False, True):
        tr = R.make_transfer(0.05, 0.0, FMAX, 0.05, 0.0, vertices=vertices)
        upd = R.HyPerLCAUpdate(ht, tr, 100.0, 1.0, True, device="cuda")
        V, A0 = torch.as_tensor(base).cuda(), torch.zeros(ht.nbatch * ht.num_ext, device="cuda")
        R.ann_activity(ht, tr, V, A0)
        Vf, Af = V.clone(), A0.clone()
        upd.update(g, V, A0)
        d.deliver(dA, None, fused=upd.args(None, Vf, Af, num_channels=1))
        torch.cuda.synchronize()
        assert torch.equal(V.view(torch.int32), Vf.view(torch.int32))
        assert torch.equal(A0.view(torch.int32), Af.view(torch.int32))
