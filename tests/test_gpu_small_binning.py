"""The library's binnings at the edges of their rules: LinkedCellList builds
around the one-workgroup sort (1, 4096, 4097, 16384, 16385 keys; up to and past
16384 bins; every key in one bin), bit-exact against numpy's stable sort; and
calls without a binning around the counting build, against the oracle."""
import numpy as np
import pytest
import torch

from test_gpu_interpolation import TOL, rel_l2

pytestmark = pytest.mark.gpu


def keys_of(pts, dims):
    c = np.minimum(np.floor(pts).astype(np.int64), np.array(dims) - 1)
    return (c[:, 0] * dims[1] + c[:, 1]) * dims[2] + c[:, 2]


@pytest.mark.parametrize("n", [1, 63, 4095, 4096, 4097, 16383, 16384, 16385])
@pytest.mark.parametrize("dims", [(3, 5, 2), (32, 16, 32), (33, 16, 32), (70, 60, 50)])
@pytest.mark.parametrize("crowded", [False, True])
def test_build_matches_a_stable_sort(ca, n, dims, crowded):
    rng = np.random.default_rng(n + sum(dims))
    pts = rng.uniform(0.0, 1.0, size=(n, 3)) * np.array(dims)
    if crowded:
        pts[n // 4:] = np.array([1.5, 0.5, 1.25])
    key = keys_of(pts, dims)
    lcl = ca.createLinkedCellList(torch.tensor(pts, device="cuda"), [1.0] * 3, [0.0] * 3,
                                  [float(d) for d in dims])
    counts = np.bincount(key, minlength=dims[0] * dims[1] * dims[2])
    assert np.array_equal(lcl.permutes.cpu().numpy(), np.argsort(key, kind="stable"))
    assert np.array_equal(lcl.counts.cpu().numpy(), counts)
    assert np.array_equal(lcl.offsets.cpu().numpy(), np.cumsum(counts) - counts)


# Tiles of 4096 keys: a ragged last one, and one past the 8192 tiles that a
# round of the digit rows' scan takes.
@pytest.mark.parametrize("n", [40961, 8192 * 4096 + 4097])
def test_tiled_sort(ca, n):
    dims = (16, 11, 9)
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.rand(n, 3, dtype=torch.float64, device="cuda", generator=g)
    x *= torch.tensor(dims, dtype=torch.float64, device="cuda")
    lcl = ca.createLinkedCellList(x, [1.0] * 3, [0.0] * 3, [float(d) for d in dims])
    c = x.floor().long()
    key = (c[:, 0] * dims[1] + c[:, 1]) * dims[2] + c[:, 2]
    assert torch.equal(lcl.permutes, torch.sort(key, stable=True).indices)
    counts = torch.bincount(key, minlength=dims[0] * dims[1] * dims[2])
    assert torch.equal(lcl.counts.long().reshape(-1), counts)


@pytest.mark.parametrize("n,cells", [(16384, 8), (16385, 8), (40000, 8), (40000, 24), (33000, 8)])
@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("cell_order", [False, True])
def test_calls_without_a_binning(ca, oracle, n, cells, order, cell_order):
    rng = np.random.default_rng(n + cells)
    pts = rng.uniform(0.0, cells, size=(n, 3))
    if cell_order:
        pts = pts[np.argsort(keys_of(pts, (cells,) * 3), kind="stable")]
    mass = rng.uniform(0.5, 1.5, size=n)
    gm = ca.createUniformGlobalMesh([0.0] * 3, [float(cells)] * 3, 1.0)
    lg = ca.createLocalGrid(ca.createGlobalGrid(gm, [True] * 3), 1)
    mesh = oracle.OMesh([0.0] * 3, [float(cells)] * 3, 1.0, halo=1)
    rho = ca.createArray("rho", ca.createArrayLayout(lg, 1, ca.Node()))
    halo = ca.createHalo(ca.NodeHaloPattern(), 1, rho)
    x = torch.tensor(pts, device="cuda")
    ca.p2g(ca.createScalarValueP2G(torch.tensor(mass, device="cuda"), 1.0), x, n, ca.Spline(order),
           halo, rho)
    ref = mesh.grid(1)
    oracle.p2g(mesh, order, 0, 1.0, pts, mass[:, None], ref)
    assert rel_l2(rho.view().cpu().numpy(), ref) < TOL[torch.float64]
    u = rng.normal(size=mesh.num_node + (3,))
    grid = ca.createArray("u", ca.createArrayLayout(lg, 3, ca.Node()))
    grid.view().copy_(torch.tensor(u))
    out = torch.zeros(n, 3, dtype=torch.float64, device="cuda")
    ca.g2p(grid, halo, x, n, ca.Spline(order), ca.createVectorValueG2P(out, 1.0))
    ref = np.zeros((n, 3))
    oracle.g2p(mesh, order, 1, 1.0, u, pts, ref)
    assert rel_l2(out.cpu().numpy(), ref) < TOL[torch.float64]


def crowd(kind, n, cells, rng):
    """Positions in random order: everywhere, in a few cells, in one, in a blob."""
    if kind == "uniform":
        return rng.uniform(0.0, cells, size=(n, 3))
    if kind == "blob":
        return np.clip(cells / 2 + 1.5 * rng.normal(size=(n, 3)), 0.0, cells - 1e-9)
    few = rng.integers(0, cells, size=(1 if kind == "one" else 3, 3))
    return few[rng.integers(0, len(few), size=n)] + rng.uniform(0.0, 1.0, size=(n, 3))


# The counting build: a crowded cell's particles share one counter, above 65536
# cells (41^3) its scan takes three launches, and it ends at 2^20 + 2^17 particles.
@pytest.mark.parametrize("kind", ["uniform", "few", "one", "blob"])
@pytest.mark.parametrize("n,cells", [(16385, 40), (70001, 41), ((1 << 20) + (1 << 17), 41),
                                     ((1 << 20) + (1 << 17) + 1, 41)])
def test_counting_build_of_crowded_clouds(ca, oracle, kind, n, cells):
    rng = np.random.default_rng(n % 1000 + cells)
    pts = crowd(kind, n, cells, rng)
    gm = ca.createUniformGlobalMesh([0.0] * 3, [float(cells)] * 3, 1.0)
    lg = ca.createLocalGrid(ca.createGlobalGrid(gm, [True] * 3), 1)
    mesh = oracle.OMesh([0.0] * 3, [float(cells)] * 3, 1.0, halo=1)
    rho = ca.createArray("rho", ca.createArrayLayout(lg, 1, ca.Node()))
    halo = ca.createHalo(ca.NodeHaloPattern(), 1, rho)
    mass = rng.uniform(0.5, 1.5, size=n)
    x = torch.tensor(pts, device="cuda")
    ca.p2g(ca.createScalarValueP2G(torch.tensor(mass, device="cuda"), 1.0), x, n, ca.Spline(1),
           halo, rho)
    ref = mesh.grid(1)
    oracle.p2g(mesh, 1, 0, 1.0, pts, mass[:, None], ref)
    own = mesh.owned_slices()
    assert rel_l2(rho.view().cpu().numpy()[own], ref[own]) < TOL[torch.float64]
    u = rng.normal(size=tuple(mesh.num_node) + (1,))
    grid = ca.createArray("u", ca.createArrayLayout(lg, 1, ca.Node()))
    grid.view().copy_(torch.tensor(u))
    out = torch.zeros(n, dtype=torch.float64, device="cuda")
    ca.g2p(grid, halo, x, n, ca.Spline(1), ca.createScalarValueG2P(out, 1.0))
    ref = np.zeros((n, 1))
    oracle.g2p(mesh, 1, 0, 1.0, u, pts, ref)
    assert rel_l2(out.cpu().numpy()[:, None], ref) < TOL[torch.float64]
