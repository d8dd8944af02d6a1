"""The FP64 cost sums at the edges of their walk over a layer's rows, against
numpy in 64 bits: rows shorter and longer than the workgroup, rows that allow
16-byte reads and rows that do not, fewer elements than threads, restricted and
extended buffers with a nonzero halo (which must not count)."""
import numpy as np
import pytest
import torch

from openpv_amd import abi, runtime as R

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1, 1, 0), (3, 5, 7, 3, 1), (2, 32, 32, 64, 2), (2, 3, 5, 1400, 1), (1, 2, 9, 4100, 1),
          (70, 4, 4, 4, 2), (1, 50, 41, 12, 3), (1, 50, 41, 12, 2)]


@pytest.mark.parametrize("shape", SHAPES)
def test_cost_sums(shape):
    rng = np.random.default_rng(5)
    l = abi.Loc.make(*shape[:4], halo=shape[4])
    for extended in (True, False):
        h = shape[4] if extended else 0
        x = rng.standard_normal((l.nbatch, l.ny + 2 * h, l.nx + 2 * h, l.nf)).astype(np.float32)
        v = x[:, h:h + l.ny, h:h + l.nx].astype(np.float64).reshape(l.nbatch, -1)
        a = np.abs(v)
        want = [(v * v).sum(1), a.sum(1),
                np.where(a < 0.75, a * (1.0 - 0.5 / 0.75 * a), 0.375).sum(1), (a > 0.5).sum(1)]
        for off in (0, 1):      # a buffer off the 16-byte boundary too
            d = torch.zeros(x.size + off, device="cuda")[off:]
            d.copy_(torch.as_tensor(x.ravel()))
            for kind, (p0, p1) in enumerate([(0, 0), (0, 0), (0.5, 0.25), (0.5, 0)]):
                got = R.cost_sum_f64(l, d, extended, kind, p0, p1).cpu().numpy()
                # sums of positive terms: n roundings of 2^-53 at most
                assert np.abs(got - want[kind]).max() <= 1e-12 * max(1.0, want[kind].max())
