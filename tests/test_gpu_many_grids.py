"""Calls of more grids than one halo launch takes (four), and of grids whose
memory interleaves (dofs of one allocation, which the halo folds and fills one
after the other), against one call per grid on arrays of their own."""
import numpy as np
import pytest
import torch

from test_gpu_interpolation import (G2P_FACTORY, P2G_FACTORY, P2G_SHAPE, TOL, rel_l2, shaped)

pytestmark = pytest.mark.gpu

CELLS = (9, 7, 8)
P2G_OPS = [0, 1, 3, 2, 4, 0, 1]
G2P_OPS = [1, 0, 4, 2, 3, 0, 1]


def setup(ca, periodic):
    high = [float(c) for c in CELLS]
    gm = ca.createUniformGlobalMesh([0.0] * 3, high, 1.0)
    lg = ca.createLocalGrid(ca.createGlobalGrid(gm, periodic), 1)
    rng = np.random.default_rng(11)
    pts = torch.tensor(rng.uniform(0.0, 1.0, size=(4000, 3)) * np.array(high), device="cuda")
    lcl = ca.createLinkedCellList(pts, [1.0] * 3, [0.0] * 3, high)
    return lg, pts[lcl.permutes].contiguous(), lcl, rng


def arrays_of(ca, lg, dofs, interleaved, dtype):
    """One array per entry, in allocations of their own or in one, dof by dof."""
    out = [ca.createArray("g", ca.createArrayLayout(lg, d, ca.Node()), dtype=dtype) for d in dofs]
    if interleaved:
        shape = tuple(out[0].view().shape[:3]) + (sum(dofs),)
        whole = torch.zeros(shape, dtype=dtype, device="cuda")
        at = 0
        for a, d in zip(out, dofs):
            a._view = whole[..., at:at + d]
            at += d
    return out


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("interleaved", [False, True])
@pytest.mark.parametrize("periodic", [[True] * 3, [True, False, True]])
@pytest.mark.parametrize("binned", [False, True])
def test_p2g_of_seven_grids(ca, binned, periodic, interleaved, dtype):
    lg, pts, lcl, rng = setup(ca, periodic)
    bins = lcl if binned else None
    n = pts.shape[0]
    dofs = [P2G_SHAPE[op][1] for op in P2G_OPS]
    fs = [getattr(ca, P2G_FACTORY[op])(
        torch.tensor(shaped(rng.normal(size=(n, P2G_SHAPE[op][0])), P2G_SHAPE[op][0]),
                     dtype=dtype, device="cuda"), 0.5) for op in P2G_OPS]
    got = arrays_of(ca, lg, dofs, interleaved, dtype)
    halo = ca.createHalo(ca.NodeHaloPattern(), 1, got[0])
    ca.p2g(fs, pts, n, ca.Spline(2), halo, got, bins=bins)
    own = lg.indexSpace(ca.Own(), ca.Node())
    box = tuple(slice(own.min(d), own.max(d)) for d in range(3))
    for f, a, d in zip(fs, got, dofs):
        one, = arrays_of(ca, lg, [d], False, dtype)
        ca.p2g(f, pts, n, ca.Spline(2), halo, one, bins=bins)
        ref = one.view()[box].cpu().numpy()
        assert rel_l2(a.view()[box].cpu().numpy(), ref) < TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("interleaved", [False, True])
@pytest.mark.parametrize("binned", [False, True])
def test_g2p_of_seven_grids(ca, binned, interleaved, dtype):
    lg, pts, lcl, rng = setup(ca, [True] * 3)
    bins = lcl if binned else None
    n = pts.shape[0]
    dofs = [{0: 1, 1: 3, 2: 1, 3: 3, 4: 3}[op] for op in G2P_OPS]
    outs = [{0: (), 1: (3,), 2: (3,), 3: (3, 3), 4: ()}[op] for op in G2P_OPS]
    grids = arrays_of(ca, lg, dofs, interleaved, dtype)
    values = [torch.tensor(rng.normal(size=tuple(a.view().shape)), dtype=dtype, device="cuda")
              for a in grids]
    for a, v in zip(grids, values):
        a.view().copy_(v)
    halo = ca.createHalo(ca.NodeHaloPattern(), 1, grids[0])

    def functors():
        out = [torch.zeros((n,) + s, dtype=dtype, device="cuda") for s in outs]
        return out, [getattr(ca, G2P_FACTORY[op])(o, 2.0) for op, o in zip(G2P_OPS, out)]

    got, fs = functors()
    ca.g2p(grids, halo, pts, n, ca.Spline(2), fs, bins=bins)
    ref, fs = functors()
    for f, v, d, a in zip(fs, values, dofs, grids):
        one, = arrays_of(ca, lg, [d], False, dtype)
        one.view().copy_(v)
        ca.g2p(one, halo, pts, n, ca.Spline(2), f, bins=bins)
        # The fill copies owners: every node of the call's grid equals this one's.
        assert torch.equal(a.view(), one.view())
    for g, r in zip(got, ref):
        assert rel_l2(g.cpu().numpy(), r.cpu().numpy()) < TOL[dtype]
