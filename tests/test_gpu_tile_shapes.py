"""Launch shapes of the stage kernels on order groups of a few elements, whose last tile is mostly
padding. The shape must not change a bit of the result: against the default shape, which the other
tests hold against the oracle."""
import numpy as np
import pytest

import ndg_cuda_amd as nd
from ndg_cuda_amd import adjoint as A
from test_gpu_stage_exchange import PULSES, grid, oblique

# order, elements of this order, elements a workgroup: the tiles need more of the RK register than the
# largest tiles do, and more than those of one element
SMALL = [(2, 13, 11), (5, 10, 3), (6, 7, 3), (6, 16, 3), (6, 6, 5), (6, 17, 5), (6, 26, 5), (8, 7, 2), (8, 5, 4), (8, 6, 4),
         (8, 13, 4), (8, 21, 4), (10, 5, 2), (10, 4, 3), (10, 10, 3), (11, 5, 2), (11, 4, 3), (11, 10, 3), (16, 3, 2)]


def run(desc, N, shapes, top=None, graph="off", steps=4):
    top = top or N
    gm = nd.Mesh2D_t(desc, N, top, 5, 0, 0, 0, 1e-6, 1e-14, 0.0, nd.NDG_t(top, 5))
    gm.initial_conditions(PULSES)
    for order, epb, remap in shapes:
        gm.set_tuning(order, epb, remap)
    assert all(s in gm.tuning() for s in shapes)
    gm.set_graph(graph)
    nd.Solver2D_t(0.5, [0.0]).run_steps(gm, steps)
    return gm


def same(a, b):
    for x, y in zip(a.get_solution(), b.get_solution()):
        assert np.array_equal(x, y)


@pytest.mark.gpu
@pytest.mark.parametrize("N,K,epb", SMALL)
@pytest.mark.parametrize("remap", [0, 1])
def test_one_group(N, K, epb, remap):
    desc = grid(K, 1, nd.BC_INFLOW, jitter=0.0)
    same(run(desc, N, [(N, epb, remap)]), run(desc, N, []))


@pytest.mark.gpu
@pytest.mark.parametrize("N", [1, 3, 8, 11, 16])
def test_tile_sizes_on_two_and_a_part(N):
    most = 64 // (N + 1)
    desc = grid(2 * most + 3, 1, nd.BC_OUTFLOW, jitter=0.0)
    ref = run(desc, N, [])
    for epb in sorted({1, 2, (most + 3) // 4, (most + 1) // 2, most - 1, most} - {0}):
        same(run(desc, N, [(N, epb, epb % 2)]), ref)


def mixed(N, K, ones):
    """`ones` elements of order 1, K of order N and, up to the largest order, 3 of order N + 1, whose register lies
    behind that of the K."""
    behind = N + 1 if N < 16 else None
    orders = np.concatenate([np.full(ones, 1), np.full(K, N), np.full(3 if behind else 0, behind or 0)])
    n = len(orders)
    desc = grid(n // 2, 2, nd.BC_INFLOW) if n % 2 == 0 else grid(n, 1, nd.BC_INFLOW, jitter=0.0)
    desc.quad_N = np.random.default_rng(K).permutation(orders).astype(np.int32)
    return desc, int(orders.max())


@pytest.mark.gpu
@pytest.mark.parametrize("N,K,epb", SMALL)
@pytest.mark.parametrize("graph", ["off", "parallel"])
def test_groups_in_one_launch(N, K, epb, graph):
    """The small group's tiles beside another group's register, in the one-launch form."""
    desc, top = mixed(N, K, 8)
    same(run(desc, 1, [(N, epb, 1)], top, graph), run(desc, 1, [], top, graph))


@pytest.mark.gpu
@pytest.mark.parametrize("N,K,epb", [(6, 6, 5), (8, 6, 4), (11, 4, 3)])
@pytest.mark.parametrize("graph", ["off", "parallel"])
def test_groups_in_a_launch_each(N, K, epb, graph):
    """As above where one element of order 1 a workgroup makes more workgroups than one launch takes: one
    launch a group, one after another and as parallel branches."""
    desc, top = mixed(N, K, 4200)
    shapes = [(1, 1, 1), (N, epb, 1)]
    same(run(desc, 1, shapes, top, graph, 2), run(desc, 1, [], top, graph, 2))


@pytest.mark.gpu
@pytest.mark.parametrize("N,n,epb", [(8, 3, 4), (8, 3, 1), (8, 3, 7), (6, 4, 3), (11, 2, 3), (16, 2, 2), (5, 3, 3)])
def test_receivers_read_the_register_of_every_shape(N, n, epb):
    """The c-derivative from the RK register at receivers in each of the elements, tile by tile."""
    desc, K = oblique(n), n * n
    rec = A.Receivers(np.arange(K), np.random.default_rng(4).uniform(-0.9, 0.9, (K, 2)))
    got = []
    for shapes in ([], [(N, epb, 0)]):
        gm = run(desc, N, shapes, steps=0)
        A.set_c_derivative(gm, "stage_records")
        got.append(A.adjoint_gradient(gm, rec, 1e-3, 6, 3))
    for a, b in zip(*got):
        assert np.array_equal(a, b)


@pytest.mark.gpu
def test_refused_shapes():
    gm = run(grid(3, 2, nd.BC_WALL), 8, [])
    for order, epb in ((8, 0), (8, 8), (7, 1)):
        with pytest.raises(nd.NDGError):
            gm.set_tuning(order, epb, 1)
    gm.set_precision("fp32c")
    with pytest.raises(nd.NDGError):  # the low words keep the order of the full tiles
        gm.set_tuning(8, 4, 1)
    gm.set_tuning(8, 7, 0)
    assert gm.tuning() == [(8, 7, 0)]
