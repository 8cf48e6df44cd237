"""What the stage kernels exchange between elements: one outgoing characteristic per side point, and
the three traces where that is not enough (periodic sides whose partner does not run parallel to
them, partners without a record), on tiles of every remainder. Against the oracle; the bar is
1e-12 in the relative maximum per field (rounding of a few steps), 2e-5 in the FP32 form."""
import numpy as np
import pytest

import ndg_cuda_amd as nd
from oracle import oracle as O

PULSES = [(0.1, -0.2, 0.4, 1.0), (-0.5, 0.4, 0.3, 0.6)]


def grid(nx, ny, bc=nd.BC_WALL, jitter=0.1, seed=3):
    """nx x ny elements on [-1, 1]^2, row by row, with jittered interior nodes; bars bottom, right,
    top, left, each along its side."""
    rng = np.random.default_rng(seed)
    X, Y = np.meshgrid(np.linspace(-1, 1, nx + 1), np.linspace(-1, 1, ny + 1), indexing="ij")
    if jitter:
        X[1:-1, 1:-1] += rng.uniform(-jitter, jitter, (nx - 1, ny - 1)) * 2 / nx
        Y[1:-1, 1:-1] += rng.uniform(-jitter, jitter, (nx - 1, ny - 1)) * 2 / ny
    n = np.arange((nx + 1) * (ny + 1)).reshape(nx + 1, ny + 1)
    i, j = (a.ravel() for a in np.meshgrid(np.arange(nx), np.arange(ny), indexing="ij"))
    quads = np.stack([n[i + 1, j], n[i + 1, j + 1], n[i, j + 1], n[i, j]], 1)
    sides = [np.stack([n[1:, 0], n[:-1, 0]], 1), np.stack([n[-1, 1:], n[-1, :-1]], 1),
             np.stack([n[:-1, -1], n[1:, -1]], 1), np.stack([n[0, :-1], n[0, 1:]], 1)]
    bars = np.concatenate(sides)
    return nd.MeshDescription(np.stack([X.ravel(), Y.ravel()], 1), quads, bars,
                              np.full(len(bars), bc, dtype=np.int32), np.full(len(bars), -1, dtype=np.int64))


def oblique(n, jitter=0.1, reciprocal=True):
    """An n x n mesh whose bottom bars are paired with the left bars and the right with the top ones (a
    quarter turn apart); not reciprocal: each bottom and right bar's donor moved on by one."""
    d = grid(n, n, nd.BC_PERIODIC, jitter)
    k = np.arange(n)
    bottom, right, top, left = k, n + k, 2 * n + k, 3 * n + k
    shift = 0 if reciprocal else 1
    d.bar_donor[left], d.bar_donor[bottom] = bottom, np.roll(left, shift)
    d.bar_donor[top], d.bar_donor[right] = right, np.roll(top, shift)
    return d


def compare(desc, N, orders=None, precision="fp64", steps=3):
    top = int(N if orders is None else np.max(orders))
    desc.quad_N = None if orders is None else np.asarray(orders, dtype=np.int32)
    tables, ndg = O.Tables(top, 5), nd.NDG_t(top, 5)
    om = O.Mesh(tables, desc, N)
    gm = nd.Mesh2D_t(desc, N, top, 5, 0, 0, 0, 1e-6, 1e-14, 0.0, ndg)
    for m in (om, gm):
        m.initial_conditions(PULSES)
    gm.set_precision(precision)
    om.run_steps(0.5, steps)
    nd.Solver2D_t(0.5, [0.0]).run_steps(gm, steps)
    bar = 1e-12 if precision == "fp64" else 2e-5
    for name, g, r in zip("puv", gm.get_solution(), om.get_state()):
        assert np.max(np.abs(g - r)) <= bar * np.max(np.abs(r)), name
    if precision == "fp64":
        om.compute_rhs(0.1)
        for name, g, r in zip("puv", gm.compute_rhs(0.1), om.get_rhs()):
            assert np.max(np.abs(g - r)) <= bar * np.max(np.abs(r)), "rhs " + name
        tr = gm.interpolate_to_boundaries()
        tr = tr.ravel() if orders is None else np.concatenate([a.ravel() for a in tr])
        assert np.max(np.abs(tr - om.get_traces())) <= bar * np.max(np.abs(tr))
    return gm, om


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
@pytest.mark.parametrize("reciprocal", [True, False])
@pytest.mark.parametrize("N", [1, 4, 8, 15, 16])
def test_oblique_periodic_sides(N, reciprocal, precision):
    compare(oblique(4, reciprocal=reciprocal), N, precision=precision)


@pytest.mark.gpu
@pytest.mark.parametrize("reciprocal", [True, False])
def test_oblique_and_unpaired_sides_with_mixed_orders(reciprocal):
    """Mortar faces that read a side without a record of its own: every side then writes its traces."""
    rng = np.random.default_rng(5)
    compare(oblique(4, reciprocal=reciprocal), 3, orders=rng.choice([3, 5, 6], 16))


@pytest.mark.gpu
def test_translated_pairs_not_reciprocal():
    """Parallel sides paired with a donor one further on: the donor's characteristic is read as it is."""
    d = grid(4, 4, nd.BC_PERIODIC, 0.1)
    k = np.arange(4)
    for s in range(4):
        d.bar_donor[4 * s + k] = 4 * ((s + 2) % 4) + np.roll(k[::-1], 1)
    compare(d, 5)


@pytest.mark.gpu
def test_oblique_sides_through_an_adaptation():
    """The device rebuild keeps the records of oblique sides, and raised neighbours make some of them mortar
    sides: the state after the adaptation steps as a mesh of the same orders does."""
    desc = oblique(4)
    ndg = nd.NDG_t(8, 5)
    gm = nd.Mesh2D_t(desc, 4, 8, 5, 0, 0, 0, 1e-3, 1e-14, 0.0, ndg)
    gm.initial_conditions(PULSES)
    assert gm.adapt(8, 0) > 0
    assert len(set(gm.orders_)) > 1
    desc.quad_N = gm.orders_.copy()
    ref = nd.Mesh2D_t(desc, 4, 8, 5, 0, 0, 0, 1e-3, 1e-14, 0.0, ndg)
    ref.set_solution(*gm.get_solution())
    for m in (gm, ref):
        nd.Solver2D_t(0.5, [0.0]).run_steps(m, 3)
    for g, r in zip(gm.get_solution(), ref.get_solution()):
        assert np.array_equal(g, r)


@pytest.mark.gpu
@pytest.mark.parametrize("N,nx,ny", [(8, 1, 1), (8, 1, 6), (8, 7, 1), (8, 8, 1), (8, 3, 5), (7, 9, 1), (7, 4, 4), (1, 31, 1),
                                     (1, 32, 1), (1, 11, 3), (2, 21, 1), (15, 1, 3), (15, 5, 1), (16, 1, 4), (16, 2, 1)])
@pytest.mark.parametrize("bc", [nd.BC_WALL, nd.BC_INFLOW])
def test_tiles_and_remainders(N, nx, ny, bc):
    compare(grid(nx, ny, bc, 0.1 if min(nx, ny) > 1 else 0.0), N)


@pytest.mark.gpu
@pytest.mark.parametrize("N", [3, 8, 11])
def test_smaller_tiles_of_the_tuner(N):
    """The tuned launch shapes give the default shape's state bit for bit (the RK register's layout
    follows the shape)."""
    desc = grid(9, 7, nd.BC_OUTFLOW)
    states = []
    for tuned in (False, True):
        gm = nd.Mesh2D_t(desc, N, N, 5, 0, 0, 0, 1e-6, 1e-14, 0.0, nd.NDG_t(N, 5))
        gm.initial_conditions(PULSES)
        if tuned:
            gm.autotune(2)
        nd.Solver2D_t(0.5, [0.0]).run_steps(gm, 4)
        states.append(gm.get_solution())
    for a, b in zip(*states):
        assert np.array_equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("N,nx,ny", [(8, 1, 1), (8, 7, 1), (8, 3, 5), (7, 9, 1), (2, 21, 1), (1, 33, 1), (11, 2, 3), (16, 2, 2)])
@pytest.mark.parametrize("bc", [nd.BC_WALL, nd.BC_INFLOW])
def test_fp32c_tiles_and_remainders(N, nx, ny, bc):
    """One element, exactly one tile, and tiles with a remainder, in the FP32 form."""
    compare(grid(nx, ny, bc, jitter=0.1 if min(nx, ny) > 1 else 0.0), N, precision="fp32c")


@pytest.mark.gpu
@pytest.mark.parametrize("bc", [nd.BC_WALL, nd.BC_INFLOW])
@pytest.mark.parametrize("orders", [(1, 2), (1, 8), (3, 4, 8), (1, 9), (5, 8, 12), (2, 13), (1, 7, 12, 16), tuple(range(1, 17))])
def test_groups_in_one_launch(orders, bc):
    """Few elements of each order: partial tiles, every kernel of the one-launch form (up to 8, 12, 16)."""
    rng = np.random.default_rng(len(orders))
    compare(grid(6, 5, bc), min(orders), orders=rng.permutation(np.resize(orders, 30)))


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny", [(260, 170), (260, 260)])
def test_groups_on_both_sides_of_the_line(nx, ny):
    """1,744 and 2,667 workgroups of two groups: one launch for both, one launch each."""
    compare(grid(nx, ny), 1, orders=np.where(np.arange(nx * ny) % nx < nx // 2, 1, 2), steps=1)


@pytest.mark.gpu
@pytest.mark.parametrize("orders", [(1, 8), (3, 4, 8), (5, 8, 12), (2, 13), tuple(range(1, 17))])
def test_fp32c_groups_in_one_launch(orders):
    rng = np.random.default_rng(len(orders))
    compare(grid(6, 5, nd.BC_INFLOW), min(orders), orders=rng.permutation(np.resize(orders, 30)), precision="fp32c")
