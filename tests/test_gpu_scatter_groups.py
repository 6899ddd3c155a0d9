"""The cell-tiled P2G scatter where its groups of equal cell go wrong: cells
of every population around its steps of 4, chunks of 16, batches of 64 and
sub-batches of 16 and 32 particles (empty ones among them), on a grid whose
extents are no multiple of a brick; particles that moved to neighbouring
cells after the binning; and values that are not finite, which must reach the
stencil nodes of their particle and no other node.  Against the oracle at the
tolerances of the other interpolation tests (FP64 1e-12, FP32-mixed 1e-5
relative L2)."""
import numpy as np
import pytest
import torch

from test_gpu_interpolation import P2G_FACTORY, P2G_SHAPE, TOL, rel_l2, shaped

pytestmark = pytest.mark.gpu

POPULATION = [0, 1, 2, 3, 4, 5, 7, 8, 9, 0, 12, 13, 15, 16, 17, 20, 31, 32, 33, 48, 63, 64, 65,
              0, 0, 130]
# 5.1 a cell, where the fused MPM P2G keeps the records of 16 particles; 3.0, where
# the FP32 one also sums groups of up to four in two chains.
SPARSE = [0, 1, 2, 3, 4, 0, 0, 16, 17, 0, 0, 1, 33, 0, 0, 5]
THIN = [0, 1, 2, 3, 4, 0, 0, 16, 17, 0, 0, 1, 0, 0, 0, 4]
CELLS = (5, 7, 19)
CELL = 0.5
LOW = np.array([0.25, -1.0, 2.0])
SETS = [(0, 1, 4), (0, 1), (0,), (1,), (2,), (3,), (4,)]


class Cloud:
    def __init__(self, ca, oracle, seed, moved=0.0, population=POPULATION):
        rng = np.random.default_rng(seed)
        cells = np.stack(np.meshgrid(*[np.arange(c) for c in CELLS], indexing="ij"), -1)
        cells = cells.reshape(-1, 3)
        pop = np.resize(population, len(cells))
        cell_of = np.repeat(cells, pop, axis=0)
        self.n = len(cell_of)
        high = LOW + CELL * np.array(CELLS)
        pts = LOW + CELL * (cell_of + rng.uniform(0.0, 1.0, size=(self.n, 3)))
        gm = ca.createUniformGlobalMesh(LOW, high, CELL)
        self.lg = ca.createLocalGrid(ca.createGlobalGrid(gm, [True] * 3), 1)
        self.mesh = oracle.OMesh(LOW, high, CELL, halo=1)
        t = torch.tensor(pts, device="cuda")
        self.bins = ca.createLinkedCellList(t, [CELL] * 3, LOW, high)
        pts = pts[self.bins.permutes.cpu().numpy()]
        if moved:
            pts = pts + moved * CELL * rng.normal(size=pts.shape)
            pts = LOW + np.mod(pts - LOW, high - LOW)
        self.pts_np = pts
        self.pts = torch.tensor(pts, device="cuda")
        self.values = {op: rng.normal(size=(self.n, P2G_SHAPE[op][0])) for op in range(5)}

    def p2g(self, ca, ops, order, dtype):
        arrays, fs = [], []
        for op in ops:
            layout = ca.createArrayLayout(self.lg, P2G_SHAPE[op][1], ca.Node())
            arrays.append(ca.createArray("g", layout, dtype=dtype))
            v = torch.tensor(shaped(self.values[op], P2G_SHAPE[op][0]), dtype=dtype, device="cuda")
            fs.append(getattr(ca, P2G_FACTORY[op])(v, -0.75))
        halo = ca.createHalo(ca.NodeHaloPattern(), 1, arrays[0])
        ca.p2g(fs, self.pts, self.n, ca.Spline(order), halo, arrays, bins=self.bins)
        assert ca.check_domain() == 0
        return [a.view().cpu().numpy() for a in arrays]

    def reference(self, oracle, op, order, dtype):
        ref = self.mesh.grid(P2G_SHAPE[op][1])
        v = self.values[op]
        if dtype == torch.float32:
            v = v.astype(np.float32).astype(np.float64)
        oracle.p2g(self.mesh, order, op, -0.75, self.pts_np, v, ref)
        return ref


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("moved", [0.0, 0.4])
@pytest.mark.parametrize("population", [POPULATION, SPARSE], ids=["dense", "sparse"])
def test_group_sizes(ca, oracle, order, dtype, moved, population):
    c = Cloud(ca, oracle, 31 + order, moved, population)
    own = c.mesh.owned_slices()
    ref = {op: c.reference(oracle, op, order, dtype) for op in range(5)}
    for ops in SETS:
        for op, got in zip(ops, c.p2g(ca, ops, order, dtype)):
            assert rel_l2(got[own], ref[op][own]) < TOL[dtype], (ops, op)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("order", [1, 2, 3])
def test_values_that_are_not_finite(ca, oracle, order, dtype):
    c = Cloud(ca, oracle, 77 + order)
    bad = [np.inf, -np.inf, np.nan]
    for op, at in ((0, 11), (1, 700), (4, 1500)):
        for k, b in enumerate(bad):
            c.values[op][at + 400 * k, -1] = b
    own = c.mesh.owned_slices()
    with np.errstate(all="ignore"):
        for op, got in zip((0, 1, 4), c.p2g(ca, (0, 1, 4), order, dtype)):
            ref = c.reference(oracle, op, order, dtype)[own]
            fine = np.isfinite(ref)
            assert not fine.all() and fine.mean() > 0.3
            assert np.array_equal(fine, np.isfinite(got[own]))
            assert rel_l2(got[own][fine], ref[fine]) < TOL[dtype]


@pytest.mark.parametrize("terms", [(0,), (1,), (0, 1), (0, 1, 4)])
@pytest.mark.parametrize("order", [1, 2])
def test_fp32_value_sums_span_eight_particles(ca, order, terms):
    """16 particles at one point whose weights are powers of two (times three):
    the first of value 2^24, the last eight of value 1.  FP32 sums of eight
    particles and FP64 sums of those are exact, and 2^24 + 8 is an FP32 number;
    one FP32 chain of 16 would lose the eight ones."""
    lg = ca.createLocalGrid(ca.createGlobalGrid(
        ca.createUniformGlobalMesh([0.0] * 3, [8.0] * 3, 1.0), [True] * 3), 1)
    at = 3.5 if order == 1 else 4.0
    pts = torch.full((16, 3), at, dtype=torch.float64, device="cuda")
    v = torch.zeros(16, 9, dtype=torch.float32, device="cuda")
    v[0], v[8:] = 2.0 ** 24, 1.0
    arrays, fs = [], []
    for op in terms:
        n, dofs = P2G_SHAPE[op]
        arrays.append(ca.createArray("g", ca.createArrayLayout(lg, dofs, ca.Node()),
                                     dtype=torch.float32))
        value = torch.zeros_like(v) if op == 4 else v[:, :n].contiguous()
        value = value.reshape((16,) if n == 1 else (16, 3) if n == 3 else (16, 3, 3))
        fs.append(getattr(ca, P2G_FACTORY[op])(value, 1.0))
    halo = ca.createHalo(ca.NodeHaloPattern(), 1, arrays[0])
    bins = ca.createLinkedCellList(pts, [1.0] * 3, [0.0] * 3, [8.0] * 3)
    ca.p2g(fs, pts, 16, ca.Spline(order), halo, arrays, bins=bins)
    w = torch.tensor([0.5, 0.5] if order == 1 else [0.125, 0.75, 0.125], dtype=torch.float64)
    sums = (2.0 ** 24 + 8.0) * w[:, None, None] * w[:, None] * w
    lo = 4  # ghosted index of the stencil's first node
    box = slice(lo, lo + len(w))
    for op, a in zip(terms, arrays):
        got = a.view()[box, box, box].double().cpu()
        for d in range(got.shape[-1] if op != 4 else 0):
            # (27 (2^24 + 8) / 64 and the like need one more rounding.)
            assert torch.all((got[..., d] - sums).abs() <= sums * 2.0 ** -24), (op, d)


@pytest.mark.parametrize("order", [1, 2, 3])
def test_large_fp32_values_keep_the_fp64_window(ca, oracle, order):
    """Values about 2^100 in crowded cells.  A node gets at most nine windows'
    sums, each rounded to FP32 (2^-24), besides the roundings of the FP32
    products and chains (2^-23): 12 * 2^-24.  One FP32 atomic a particle and
    node would round thousands of times."""
    c = Cloud(ca, oracle, 5, population=[200])
    c.values[0] = np.float32(np.abs(c.values[0]) + 0.5).astype(np.float64) * 2.0 ** 100
    own = c.mesh.owned_slices()
    got, = c.p2g(ca, (0,), order, torch.float32)
    ref = c.reference(oracle, 0, order, torch.float32)
    assert rel_l2(got[own] * 2.0 ** -100, ref[own] * 2.0 ** -100) < 12 * 2.0 ** -24


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("moved", [0.05, 0.15, 0.6])
@pytest.mark.parametrize("population", [POPULATION, SPARSE], ids=["dense", "sparse"])
def test_positions_that_moved_since_the_binning(ca, oracle, order, dtype, moved, population):
    """Batches whose cells are out of order are taken in cell order, and particles
    of a quadratic spline up to half a cell out of their row keep its window: P2G
    against the oracle, the G2P adjoint against the per-particle kernels."""
    c = Cloud(ca, oracle, 57 + order, moved, population)
    own = c.mesh.owned_slices()
    for op, got in zip((0, 1, 4), c.p2g(ca, (0, 1, 4), order, dtype)):
        assert rel_l2(got[own], c.reference(oracle, op, order, dtype)[own]) < TOL[dtype], op
    rng = np.random.default_rng(3)
    vbar = torch.tensor(rng.normal(size=(c.n, 3)), dtype=dtype, device="cuda")
    lbar = torch.tensor(rng.normal(size=(c.n, 3, 3)), dtype=dtype, device="cuda")
    u, ubar, uref = (ca.createArray("u", ca.createArrayLayout(c.lg, 3, ca.Node()), dtype=dtype)
                     for _ in range(3))
    halo = ca.createHalo(ca.NodeHaloPattern(), 1, u)
    fs = [ca.createVectorValueG2P(vbar, 1.5), ca.createVectorGradientG2P(lbar, -0.5)]

    def adjoint(out, bins):
        ca.g2p_adjoint([u, u], halo, c.pts, c.n, ca.Spline(order), fs, [vbar, lbar], [out, out],
                       None, bins=bins)

    adjoint(ubar, c.bins)
    ca.set_auto_binning(False)
    try:
        adjoint(uref, None)
    finally:
        ca.set_auto_binning(True)
    assert rel_l2(ubar.view().cpu().numpy()[own], uref.view().cpu().numpy()[own]) < TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("moved", [0.0, 0.15])
def test_thin_clouds(ca, oracle, order, dtype, moved):
    c = Cloud(ca, oracle, 91 + order, moved, THIN)
    own = c.mesh.owned_slices()
    for ops in SETS:
        for op, got in zip(ops, c.p2g(ca, ops, order, dtype)):
            ref = c.reference(oracle, op, order, dtype)
            assert rel_l2(got[own], ref[own]) < TOL[dtype], (ops, op)
