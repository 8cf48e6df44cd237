"""Sides that do not quite lie on one line: the faces of a hanging side up to the topology's tolerance (1e-12 of
its length) off it, and periodic pairs a little out of parallel. Each face's flux has its own direction and
each periodic side its own normal, as the oracle's. The bar: a right-hand side of random values sums some
2 (N+1) + 4 terms of its own size, at most 30 roundings of 1.1e-16 and as many in the oracle, 7e-15 in
all; 4e-14 leaves room for terms larger than their sum and is a twentieth of the directions' difference here."""
import numpy as np
import pytest

import ndg_cuda_amd as nd
from meshes import split_elements
from oracle import oracle as O
from test_gpu_stage_exchange import PULSES, grid


def rhs_of(desc, N, top):
    tables, ndg = O.Tables(top, 5), nd.NDG_t(top, 5)
    om = O.Mesh(tables, desc, N)
    gm = nd.Mesh2D_t(desc, N, top, 5, 0, 0, 0, 1e-6, 1e-14, 0.0, ndg)
    rng = np.random.default_rng(11)
    q = [rng.standard_normal(gm.n_dofs_per_field_) for _ in range(3)]
    gm.set_solution(*q)
    om.set_state(*q)
    om.compute_rhs(0.1)
    return gm, gm.compute_rhs(0.1), om.get_rhs()


def off_the_line(desc, off):
    """The nodes halfway along an edge that no other element and no bar has, moved across it by +- off of its
    length; returns how many."""
    quads = np.asarray(desc.quads)
    edges = {(int(q[s]), int(q[(s + 1) % 4])) for q in quads for s in range(4)}
    bars = {frozenset(map(int, b)) for b in np.asarray(desc.bars)}
    n = 0
    for a, b in sorted(edges):
        if (b, a) in edges or frozenset((a, b)) in bars:
            continue
        pa, pb = desc.xy[a], desc.xy[b]
        d = np.hypot(*(desc.xy - (pa + pb) / 2).T)
        m = int(np.argmin(d))
        if d[m] > 1e-9:
            continue  # a half of such an edge
        desc.xy[m] += (off if n % 2 else -off) * np.array([-(pb - pa)[1], (pb - pa)[0]])
        n += 1
    return n


@pytest.mark.gpu
@pytest.mark.parametrize("more", [(), (1, 4)])
@pytest.mark.parametrize("N", [1, 2, 5, 8])
def test_hanging_faces_off_the_side(N, more):
    desc = grid(5, 5, nd.BC_WALL, 0.1)
    if more:
        desc.quad_N = np.random.default_rng(2).choice([N, *(N + k for k in more)], 25).astype(np.int32)
    desc = split_elements(desc, [6, 12, 13])
    assert off_the_line(desc, 0.8e-12) >= 6
    gm, got, want = rhs_of(desc, N, N + max(more, default=0))
    for name, g, r in zip("puv", got, want):
        assert np.max(np.abs(g - r)) <= 4e-14 * np.max(np.abs(r)), name


def nearly_periodic(n, turn, seed):
    """An n x n mesh of translated periodic pairs; the inner nodes of the bottom and left boundary moved off it so
    that the pairs are out of parallel by about `turn`."""
    d = grid(n, n, nd.BC_PERIODIC, 0.1)
    k = np.arange(n)
    for s in range(4):
        d.bar_donor[n * s + k] = n * ((s + 2) % 4) + k
    rng = np.random.default_rng(seed)
    for axis in (0, 1):  # across the side at coordinate -1 of the axis
        on = np.flatnonzero((d.xy[:, axis] == -1) & (np.abs(d.xy[:, 1 - axis]) < 0.99))
        d.xy[on, axis] += rng.choice([-0.5, 0.5], len(on)) * turn * 2 / n
    return d


@pytest.mark.gpu
@pytest.mark.parametrize("turn", [0.8e-12, 1e-13, 0.0])
@pytest.mark.parametrize("N", [1, 2, 5, 8])
def test_periodic_pairs_out_of_parallel(N, turn):
    gm, got, want = rhs_of(nearly_periodic(6, turn, 3), N, N)
    for name, g, r in zip("puv", got, want):
        assert np.max(np.abs(g - r)) <= 4e-14 * np.max(np.abs(r)), name


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["device", "host"])
def test_periodic_pairs_out_of_parallel_through_an_adaptation(mode):
    """Both rebuilds judge the new sides by their own vertices, as a mesh made of them does."""
    desc = nearly_periodic(4, 0.8e-12, 4)
    ndg = nd.NDG_t(8, 5)
    gm = nd.Mesh2D_t(desc, 4, 8, 5, 0, 0, 0, 1e-3, 1e-14, 0.0, ndg)
    gm.initial_conditions(PULSES)
    gm.set_adapt_mode(mode)
    assert gm.adapt(8, 0) > 0
    desc.quad_N = gm.orders_.copy()
    ref = nd.Mesh2D_t(desc, 4, 8, 5, 0, 0, 0, 1e-3, 1e-14, 0.0, ndg)
    ref.set_solution(*gm.get_solution())
    for g, r in zip(gm.compute_rhs(0.0), ref.compute_rhs(0.0)):
        assert np.array_equal(g, r)
