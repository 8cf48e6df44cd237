"""The estimator on element counts around its workgroup tiles (85 elements of order 1, 17 of order 3, 8 of order 8, 5
of order 12, 4 of order 16), on a random state: error estimates to 1e-12 relative, the decay rate sigma to 1e-8 (a
log-fit of sums that cancel by a few digits), the same flags as the oracle."""
import numpy as np
import pytest

import ndg_cuda_amd as nd
from oracle import oracle as O
from test_gpu_stage_exchange import grid


@pytest.mark.gpu
@pytest.mark.parametrize("N,K", [(1, 1), (1, 84), (1, 85), (1, 86), (3, 17), (3, 18), (8, 1), (8, 7), (8, 8), (8, 9), (12, 5),
                                 (16, 1), (16, 3), (16, 4), (16, 5)])
def test_estimator_tiles(N, K):
    desc = grid(K, 1, nd.BC_WALL, 0.0)
    gm = nd.Mesh2D_t(desc, N, N, 5, 0, 0, 0, 1e-6, 1e-14, 0.0, nd.NDG_t(N, 5))
    om = O.Mesh(O.Tables(N, 5), desc, N)
    rng = np.random.default_rng(N * 100 + K)
    q = [rng.standard_normal(gm.n_dofs_per_field_) for _ in range(3)]
    gm.set_solution(*q)
    om.set_state(*q)
    eg, sg, rg, cg = gm.estimate_error()
    eo, so, ro, co = om.estimate_error()
    assert np.max(np.abs(eg - eo) / np.abs(eo)) < 1e-12
    assert np.max(np.abs(sg - so) / np.abs(so)) < 1e-8
    assert np.array_equal(rg, ro) and np.array_equal(cg, co)
