"""Host reads allocate no device memory (GPU)."""
from __future__ import annotations

import pytest

import cudadsmc_amd as dm

from helpers import small_physics_settings

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _solver(dims, n, seed=1, grid=None):
    s = small_physics_settings(dims=dims, n_target=n)
    s.seed = seed
    sol = dm.Solver()
    sol.Init(s)
    sol.SetModel(dm.icosphere((0.07, 0.05, 0.05), 0.02, 2), grid=(8, 8, 8))
    sol.InitSystemState(tuple(s.stream_velocity))
    if grid:
        sol.set_scatter_grid(grid)
    return sol


def _free() -> int:
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def test_reads_allocate_no_device_memory():
    warm = _solver((16, 12, 12), 20000)  # what a kernel's first launch sets up is not meant
    for _ in range(2):
        warm.set_sampling(True)
        warm.DoBenchmark(3, warm.settings.dt)
        warm.fields(), warm.drag(), warm.cell_stats(), warm.collision_stats()
    sol = _solver((128, 64, 64), 50000)
    sol.DoBenchmark(3, sol.settings.dt)
    sol.synchronize()
    before = _free()
    sol.set_sampling(True)
    sol.fields(), sol.drag(), sol.cell_stats(), sol.collision_stats()
    assert before - _free() < 20 * sol.n_cells  # the fields on their way to the host: 20 bytes per cell
    sol.close()
    warm.close()
