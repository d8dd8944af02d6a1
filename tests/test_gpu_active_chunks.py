"""The active list where its chunking changes: layers of one round per chunk up
to the number of chunks that takes in one image and in the batch, the 16-round
chunks beyond, several counts per thread of the scan, odd extended sizes, and
empty and full buffers."""
import numpy as np
import pytest
import torch

from openpv_amd import abi, runtime as R

pytestmark = pytest.mark.gpu

SHAPES = [  # nbatch, nx, ny, nf, halo; density
    ((1, 1, 1, 3, 0), 0.5), ((2, 13, 11, 7, 1), 0.3), ((5, 30, 20, 64, 2), 0.07),
    ((1, 128, 128, 512, 0), 0.02), ((1, 129, 128, 512, 0), 0.02),
    ((1, 128, 128, 448, 0), 0.02),      # 7168 chunks of one round, seven per thread of the scan
    ((1, 129, 128, 448, 0), 0.02),      # one more column: chunks of 16 rounds
    ((2, 128, 128, 256, 0), 0.02),      # 8192 in the batch
    ((2, 129, 128, 256, 0), 0.02),      # ... and beyond
    ((2, 64, 64, 100, 0), 0.0), ((1, 64, 64, 100, 1), 1.0), ((300, 5, 5, 9, 1), 0.2),
]


@pytest.mark.parametrize("case", SHAPES)
def test_active_list(case):
    (nb, nx, ny, nf, halo), density = case
    l = abi.Loc.make(nb, nx, ny, nf, halo=halo)
    g = torch.Generator(device="cuda").manual_seed(6)
    a = torch.randn(nb * l.num_ext, device="cuda", generator=g)
    a[torch.rand(a.shape, device="cuda", generator=g) >= density] = 0
    al = R.ActiveList(l, torch.device("cuda"))
    al.compact(a)
    torch.cuda.synchronize()
    ent, num = al.host_entries()
    pos = al.pos_start.cpu().numpy().reshape(nb, -1)
    A = a.cpu().numpy().reshape(nb, -1)
    for b in range(nb):
        idx = np.flatnonzero(A[b])
        assert num[b] == len(idx)
        assert np.array_equal(ent[b, :len(idx)]["index"], idx)
        assert np.array_equal(ent[b, :len(idx)]["value"], A[b][idx])
        want = np.searchsorted(idx, np.arange(l.nx_ext * l.ny_ext + 1) * nf)
        assert np.array_equal(pos[b], want)
