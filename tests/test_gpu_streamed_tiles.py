"""The stages of a mesh whose state is streamed past the caches (more than 242 MB a stage), on tiles that start
inside a 128-byte line, end inside a 16-byte word or hold an odd number of line indices: many unconnected
copies of a small mesh must step as the small mesh, which stays in the caches, bit for bit."""
import numpy as np
import pytest

import ndg_cuda_amd as nd
from test_gpu_stage_exchange import PULSES, grid


def copies(desc, n):
    """n times the same elements on nodes and bars of their own: 65 elements are no multiple of a tile, so that the
    copies meet the tiles at every place."""
    nodes, K = len(desc.xy), len(desc.quads)
    at = np.arange(n)[:, None, None] * nodes
    return nd.MeshDescription(np.tile(desc.xy, (n, 1)), (desc.quads[None] + at).reshape(n * K, 4),
                              (desc.bars[None] + at).reshape(-1, 2), np.tile(desc.bar_type, n),
                              np.full(n * len(desc.bars), -1, dtype=np.int64))


@pytest.mark.gpu
@pytest.mark.parametrize("precision,N", [("fp64", 8), ("fp64", 12), ("fp64", 16), ("fp32c", 8), ("fp32c", 12), ("fp32c", 4)])
def test_copies_of_a_small_mesh(N, precision):
    small = grid(13, 5, nd.BC_WALL)
    values = 65 * 3 * (N + 1) ** 2
    n = 260000000 // ((16 if precision == "fp64" else 12) * values) + 2
    states = []
    for desc in (small, copies(small, n)):
        gm = nd.Mesh2D_t(desc, N, N, 5, 0, 0, 0, 1e-6, 1e-14, 0.0, nd.NDG_t(N, 5))
        gm.initial_conditions(PULSES)
        gm.set_precision(precision)
        nd.Solver2D_t(0.5, [0.0]).run_steps(gm, 2)
        states.append(gm.get_solution())
    for one, all_ in zip(*states):
        assert np.array_equal(all_.reshape(n, -1), np.broadcast_to(one, (n, one.size)))
