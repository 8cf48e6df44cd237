"""Reading from a mesh between steps leaves the run as it is, bit for bit."""
import numpy as np
import pytest

import ndg_cuda_amd as nd
from test_gpu_stage_exchange import PULSES, grid, oblique


def runs(desc, N, top=None, orders=None, precision="fp64", graph="off"):
    """The state after eight steps, without and with reads of the traces, right-hand side and estimate between them."""
    top = top or N
    desc.quad_N = None if orders is None else np.asarray(orders, dtype=np.int32)
    for read in (False, True):
        gm = nd.Mesh2D_t(desc, N, top, 5, 0, 0, 0, 1e-6, 1e-14, 0.0, nd.NDG_t(top, 5))
        gm.initial_conditions(PULSES)
        gm.set_precision(precision)
        gm.set_graph(graph)
        solver, time = nd.Solver2D_t(0.5, [0.0]), 0.0
        for _ in range(4):
            time = solver.run_steps(gm, 2, time)
            if read:
                first = gm.interpolate_to_boundaries()
                gm.compute_rhs(time)
                gm.estimate_error()
                for a, b in zip(first, gm.interpolate_to_boundaries()):
                    assert np.array_equal(a, b)
        yield gm.get_solution()


@pytest.mark.gpu
@pytest.mark.parametrize("bc", [nd.BC_WALL, nd.BC_INFLOW, nd.BC_PERIODIC])
@pytest.mark.parametrize("N", range(1, 17))
def test_reads_between_steps(N, bc):
    desc = oblique(4) if bc == nd.BC_PERIODIC else grid(5, 3, bc)
    for a, b in zip(*runs(desc, N)):
        assert np.array_equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
@pytest.mark.parametrize("graph", ["off", "sequential", "parallel"])
def test_reads_between_steps_of_mixed_orders(graph, precision):
    orders = np.random.default_rng(7).choice([2, 4, 5, 8], 30)
    for a, b in zip(*runs(grid(6, 5, nd.BC_INFLOW), 2, 8, orders, precision, graph)):
        assert np.array_equal(a, b)
