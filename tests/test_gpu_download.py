"""Large downloads, which pass through pinned slots in pieces that cut elements and planes anywhere, give the
values bit for bit in the caller's order."""
import numpy as np
import pytest

import ndg_cuda_amd as nd
from ndg_cuda_amd._abi import lib
from test_gpu_stage_exchange import grid


def make(nx, ny, top, orders=None, n_points=5):
    desc = grid(nx, ny, nd.BC_WALL)
    if orders is not None:
        desc.quad_N = np.asarray(orders, dtype=np.int32)
    first = top if orders is None else int(np.min(orders))
    return nd.Mesh2D_t(desc, first, top, n_points, 0, 0, 0, 1e-6, 1e-14, 0.0, nd.NDG_t(top, n_points))


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny,top,mixed", [(66, 66, 8, False), (66, 65, 8, False), (150, 97, 9, True), (200, 113, 8, True), (113, 113, 8, False)])
def test_state_round_trip(nx, ny, top, mixed):
    """Below and above the line between the two ways, up to five slots' worth, elements of several sizes."""
    rng = np.random.default_rng(7)
    m = make(nx, ny, top, rng.integers(1, top + 1, nx * ny) if mixed else None)
    state = [rng.standard_normal(m.n_dofs_per_field_) for _ in range(3)]
    m.set_solution(*state)
    for _ in range(2):
        for a, b in zip(state, m.get_solution()):
            assert np.array_equal(a, b)
    out = np.empty_like(state[1])  # fields without a place are left out
    assert lib().ndg_get_state(m._h, None, out.ctypes.data, None) == 0
    assert np.array_equal(out, state[1])


@pytest.mark.gpu
def test_output_planes():
    """Planes one by one (small downloads) and several at once (large ones) are the same bits."""
    m = make(70, 61, 4, n_points=8)
    rng = np.random.default_rng(9)
    m.set_solution(*(rng.standard_normal(m.n_dofs_per_field_) for _ in range(3)))
    n = 70 * 61 * 8 * 8

    def planes(wanted):
        out = [np.full(n, np.nan) if k in wanted else None for k in range(5)]
        assert lib().ndg_get_solution(m._h, *(None if a is None else a.ctypes.data for a in out)) == 0
        return out

    single = [planes({k})[k] for k in range(5)]
    for wanted in ({0, 1, 2, 3, 4}, {0, 2, 3, 4}, {1, 2, 3, 4}):
        for k, a in enumerate(planes(wanted)):
            assert (a is None) == (k not in wanted) and (a is None or np.array_equal(a, single[k]))
