"""The size of the RK register against every tile size that a stage launch may take (host code only)."""
import ctypes

import pytest

from ndg_cuda_amd import _abi


@pytest.mark.parametrize("N", range(1, 17))
def test_rk_register_holds_tiles_of_every_size(N):
    """Tile b of `epb` elements lies at 3 (N+1) run values a tile, a last partial tile at full length: all tiles
    end within the values that the register has for K elements."""
    L = _abi.lib()
    run = getattr(L, "_ZN3ndg9stage_runEii")                # int ndg::stage_run(int N, int epb)
    values = getattr(L, "_ZN3ndg15stage_rk_valuesEil")      # int64_t ndg::stage_rk_values(int N, int64_t K)
    run.argtypes, run.restype = [ctypes.c_int, ctypes.c_int], ctypes.c_int
    values.argtypes, values.restype = [ctypes.c_int, ctypes.c_int64], ctypes.c_int64
    most = 64 // (N + 1)
    runs = {epb: run(N, epb) for epb in range(1, most + 1)}
    assert all(r >= epb * (N + 1) for epb, r in runs.items())
    for K in list(range(1, most * most * 4 + 2)) + [4095, 4096, 4097, 262144]:
        for epb, r in runs.items():
            assert -(-K // epb) * 3 * (N + 1) * r <= values(N, K), (N, K, epb)
