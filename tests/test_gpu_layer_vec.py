"""The 16-byte forms of the layer updates and of the transfer give the bits of
the element-wise forms (which the oracle tests pin): the same call on buffers
one value off the 16-byte boundary runs those.  Images at the 1024 neurons the
16-byte form starts at (smaller ones are element-wise either way) and layers
that end inside a workgroup, one and several channels, A(t-1) read and
recomputed (for ISTA from 2^18 neurons on), the chunked BF16 copy, and A left
out."""
import numpy as np
import pytest
import torch

from openpv_amd import abi, runtime as R

pytestmark = pytest.mark.gpu
FMAX = float(np.finfo(np.float32).max)
SHAPES = [(1, 1, 1, 4, 0), (2, 5, 3, 12, 1), (3, 16, 9, 64, 2), (1, 6, 2, 2, 2), (2, 33, 17, 32, 3),
          (2, 16, 16, 4, 0), (1, 6, 171, 2, 2), (3, 7, 37, 4, 0), (2, 43, 19, 12, 1), (1, 17, 15, 4, 2),
          (2, 64, 57, 36, 1)]


def at(x, off):
    """x in a buffer `off` values past a 16-byte boundary."""
    d = torch.zeros(x.numel() + 4, device="cuda")[off:off + x.numel()]
    d.copy_(x)
    return d


def same(a, b):
    return torch.equal(a.view(torch.int32), b.view(torch.int32))


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("rule", ["lca", "momentum", "ista"])
def test_update_bits(shape, rule):
    g = torch.Generator().manual_seed(3)
    l = abi.Loc.make(*shape[:4], halo=shape[4])
    n, ne = l.nbatch * l.num_res, l.nbatch * l.num_ext
    rnd = lambda k: 0.2 * torch.randn(k, generator=g)
    V, A, prev = rnd(n), rnd(ne), rnd(n)
    for coeffs in ((1.0,), (1.0, -0.5)):
        G = rnd(n * len(coeffs))
        for from_v in (True, False):
            for vertices in (False, True):
                t = R.make_transfer(0.1, 0.0, FMAX, 0.05, 0.03, vertices)
                out = []
                for off in (0, 1):
                    args = dict(timeConstantTau=10.0, dt=1.0, channel_coeffs=coeffs, activity_from_v=from_v)
                    if rule == "momentum":
                        u = R.MomentumLCAUpdate(l, t, LCAMomentumRate=0.3, **args)
                        u.prev_drive = at(prev, off)
                    elif rule == "ista":
                        u = R.ISTAUpdate(l, t, 0.1, **args)
                    else:
                        u = R.HyPerLCAUpdate(l, t, **args)
                    v, a = at(V, off), at(A, off)
                    b16 = R.bf16c_buffer(l) if l.nf % 32 == 0 else None
                    u.update(at(G, off), v, a, A_bf16c=b16)
                    res = [v, a] + ([u.prev_drive] if rule == "momentum" else [])
                    if b16 is not None:
                        res.append(b16.view(torch.int32))
                        if from_v and rule == "lca":    # only the copy written
                            v2 = at(V, off)
                            b2 = R.bf16c_buffer(l)
                            u.update(at(G, off), v2, None, A_bf16c=b2)
                            res += [v2, b2.view(torch.int32)]
                    out.append(res)
                torch.cuda.synchronize()
                for x, y in zip(*out):
                    assert same(x.contiguous(), y.contiguous())


@pytest.mark.parametrize("shape", SHAPES)
def test_activity_bits(shape):
    l = abi.Loc.make(*shape[:4], halo=shape[4])
    V = torch.randn(l.nbatch * l.num_res, generator=torch.Generator().manual_seed(4))
    t = R.make_transfer(0.1, 0.0, 1.5, 0.05, 0.03)
    out = []
    for off in (0, 1):
        a = at(torch.full((l.nbatch * l.num_ext,), 7.0), off)
        R.ann_activity(l, t, at(V, off), a)
        out.append(a)
    torch.cuda.synchronize()
    assert same(*out)
