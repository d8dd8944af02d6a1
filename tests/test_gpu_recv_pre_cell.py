"""The cell form of the sparse scatter (a target t times finer, one data patch
per source feature) against the oracle, at the edges of its tiling: every
number of targets per thread, cells cut by both sides of the target, the
staged weights split by column class, one wave per workgroup and several
whose items are sorted, lists that start at odd entries, empty rows, a list
that fills its buffer, and the geometries beside it that keep the other
kernels."""
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
    ((2, 33, 18, 48, 2), (2, 132, 72, 1, 0), 16, 0.07),  # t 4, four; ten workgroups per class
    ((3, 6, 5, 64, 2), (3, 24, 20, 2, 0), 12, 0.2),      # t 4, eight
    ((1, 4, 3, 512, 2), (1, 16, 12, 3, 0), 16, 0.05),    # t 4, weights of one column class at a time
    ((1, 8, 8, 32, 2), (1, 32, 32, 1, 0), 16, 1.0),      # every neuron active, halo too: a full list
    ((1, 5, 3, 7, 1), (1, 10, 6, 1, 0), 6, 0.5),         # odd extended size: another kernel
    ((70, 3, 3, 10, 1), (70, 6, 6, 1, 0), 4, 0.02),      # nearly empty lists, many batch elements
]

# A workgroup of several waves sorts its items by list length.  With batch
# elements times row and column classes at or above the 512 workgroups wanted
# (256 where the weights take more than 80 KB) it owns the whole of its class.
SORTED = [
    # pre, post, patch; items of a class, threads of a workgroup
    ((300, 9, 9, 8, 1), (300, 18, 18, 1, 0), 4),      # 90 items on 128 threads
    ((100, 20, 20, 6, 1), (100, 40, 40, 1, 0), 6),    # 420 in three workgroups of 192
    ((256, 48, 48, 2, 1), (256, 96, 96, 1, 0), 4),    # 2352 on 1024: sorted in two passes
    ((64, 10, 8, 512, 2), (64, 40, 32, 1, 0), 16),    # 139 KB of weights; 88 on 128
    ((180, 11, 8, 5, 1), (180, 33, 24, 1, 0), 9),     # odd extended width, t 3: V = 3
    ((130, 12, 13, 10, 1), (130, 24, 26, 3, 0), 4),   # V = 6
    ((140, 9, 10, 12, 1), (140, 36, 40, 2, 0), 8),    # V = 8
]


@pytest.mark.parametrize("case", CASES)
def test_cell_scatter_equals_oracle(case):
    pt, qt, p, dens = case
    rng = np.random.default_rng(71)
    hp = abi.Loc.make(*pt[:4], halo=pt[4])
    W = (rng.standard_normal((hp.nf, p, p, qt[3])) * 0.1).astype(np.float32)
    A = rng.standard_normal(hp.nbatch * hp.num_ext).astype(np.float32)
    A[rng.random(A.shape) >= dens] = 0          # the halo's neurons are active too
    check(rng, pt, qt, p, W, A)


@pytest.mark.parametrize("case", SORTED)
def test_cell_scatter_of_sorted_items_equals_oracle(case):
    pt, qt, p = case
    rng = np.random.default_rng(72)
    hp = abi.Loc.make(*pt[:4], halo=pt[4])
    W = (rng.standard_normal((hp.nf, p, p, qt[3])) * 0.1).astype(np.float32)
    # list lengths from empty to full: the active share falls from 1 at one
    # corner to 0 well before the other, and every seventh image is empty
    y, x = np.mgrid[0:hp.ny_ext, 0:hp.nx_ext]
    share = np.clip(1.0 - 1.5 * (x / hp.nx_ext + y / hp.ny_ext) / 2, 0, 1) ** (3 if hp.nf > 100 else 1)
    A = rng.standard_normal((hp.nbatch, hp.ny_ext, hp.nx_ext, hp.nf)).astype(np.float32)
    A[rng.random(A.shape, dtype=np.float32) >= share[None, :, :, None]] = 0
    A[::7] = 0
    check(rng, pt, qt, p, W, A.ravel())


def check(rng, pt, qt, p, W, A):
    hp, op = abi.Loc.make(*pt[:4], halo=pt[4]), O.Loc.make(*pt[:4], halo=pt[4])
    hq, oq = abi.Loc.make(*qt[:4], halo=qt[4]), O.Loc.make(*qt[:4], halo=qt[4])
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
