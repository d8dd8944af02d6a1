"""The cell form of the sparse scatter (a target t times finer, one data patch
per source feature) against the oracle, at the edges of its tiling: every
number of targets per thread, cells cut by both sides of the target, the
staged weights split by column class, one wave and several sorted items per
workgroup, lists that start at odd entries, empty rows, a list that fills its
buffer, and the geometries beside it that keep the other kernels."""
import numpy as np
import pytest
import torch

import oracle as O
from openpv_amd import abi, runtime as R

pytestmark = pytest.mark.gpu
DEV = "cuda"

CASES = [
    # pre (nbatch, nx, ny, nf, halo), post, patch, density
    ((2, 9, 7, 6, 1), (2, 9, 7, 1, 0), 3, 0.4),          # t 1, one target per thread
    ((1, 5, 6, 12, 2), (1, 5, 6, 3, 1), 5, 0.5),         # t 1, three
    ((1, 64, 32, 24, 4), (1, 128, 64, 1, 0), 18, 0.4),   # t 2, two; one wave per workgroup
    ((2, 7, 9, 20, 1), (2, 14, 18, 3, 2), 6, 0.3),       # t 2, six
    ((1, 11, 5, 16, 1), (1, 33, 15, 1, 0), 9, 0.6),      # t 3, three; odd patch
    ((2, 33, 18, 48, 2), (2, 132, 72, 1, 0), 16, 0.07),  # t 4, four; more items than threads
    ((3, 6, 5, 64, 2), (3, 24, 20, 2, 0), 12, 0.2),      # t 4, eight
    ((1, 4, 3, 512, 2), (1, 16, 12, 3, 0), 16, 0.05),    # t 4, weights of one column class at a time
    ((1, 8, 8, 32, 2), (1, 32, 32, 1, 0), 16, 1.0),      # every neuron active, halo too: a full list
    ((1, 5, 3, 7, 1), (1, 10, 6, 1, 0), 6, 0.5),         # odd extended size: another kernel
    ((70, 3, 3, 10, 1), (70, 6, 6, 1, 0), 4, 0.02),      # nearly empty lists, many batch elements
]


@pytest.mark.parametrize("case", CASES)
def test_cell_scatter_equals_oracle(case):
    rng = np.random.default_rng(71)
    (pt, qt, p, dens) = case
    hp, op = abi.Loc.make(*pt[:4], halo=pt[4]), O.Loc.make(*pt[:4], halo=pt[4])
    hq, oq = abi.Loc.make(*qt[:4], halo=qt[4]), O.Loc.make(*qt[:4], halo=qt[4])
    W = (rng.standard_normal((hp.nf, p, p, hq.nf)) * 0.1).astype(np.float32)
    A = rng.standard_normal(hp.nbatch * hp.num_ext).astype(np.float32)
    A[rng.random(A.shape) >= dens] = 0          # the halo's neurons are active too
    ent, cnt = O.active_indices(op, A)
    base = rng.standard_normal(hq.nbatch * hq.num_res).astype(np.float32)
    dW, dA = torch.as_tensor(W.ravel()).to(DEV), torch.as_tensor(A).to(DEV)
    al = R.ActiveList(hp, DEV)
    al.entries.fill_(-1)                        # whatever lies past a list
    al.compact(dA)
    for accumulate, dtf in ((False, 1.0), (True, 0.7)):
        ref = O.recv_pre(op, oq, p, p, W, entries=ent, num_active=cnt, dt_factor=dtf, num_threads=1,
                         gsyn=base.copy() if accumulate else None)
        for arith in (abi.ARITH_EXACT, abi.ARITH_FP32):
            d = R.PresynapticPerspectiveGPUDelivery(hp, hq, p, p, dW, arith=arith, dt_factor=dtf)
            d.mode = "ordered"
            g = torch.as_tensor(base).to(DEV)
            d.deliver(g, active=al, accumulate=accumulate)
            torch.cuda.synchronize()
            got = g.cpu().numpy()
            if arith == abi.ARITH_EXACT:
                assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))
            else:   # the same order, each product not rounded by itself
                assert np.abs(got - ref).max() <= 1e-5 * np.abs(ref).max()
