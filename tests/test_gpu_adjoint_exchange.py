"""The transposed right-hand side against the right-hand side, <G q, y> = <q, G^T y>, on tiles of every remainder and
with periodic sides whose partner does not run parallel to them (their exchanged value belongs to
another normal than the receiver's). The bar is 1e-12 |G q| |y| (rounding of the sums)."""
import numpy as np
import pytest

import ndg_cuda_amd as nd
from ndg_cuda_amd import adjoint as A
from test_gpu_stage_exchange import oblique


@pytest.mark.gpu
@pytest.mark.parametrize("N", range(1, 17))
@pytest.mark.parametrize("n", [2, 4])
def test_transpose(N, n):
    rng = np.random.default_rng(N)
    for desc in (nd.square_mesh(n, x_periodic=True, y_periodic=True, jitter=0.1, seed=2), oblique(n + 1)):
        m = nd.Mesh2D_t(desc, N, N, 5, 0, 0, 0, 1e-6, 1e-14, 0.0, nd.NDG_t(N, 5))
        q, y = ([rng.standard_normal(m.n_dofs_per_field_) for _ in range(3)] for _ in range(2))
        m.set_solution(*q)
        Gq, Gty = np.concatenate(m.compute_rhs(0.0)), np.concatenate(A.apply_rhs_transpose(m, *y))
        q, y = np.concatenate(q), np.concatenate(y)
        assert abs(Gq @ y - q @ Gty) <= 1e-12 * np.linalg.norm(Gq) * np.linalg.norm(y)
