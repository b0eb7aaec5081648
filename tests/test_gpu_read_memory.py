"""Host reads and batched steps allocate no device memory, and a batch follows
the scatter grids of its members (GPU)."""
from __future__ import annotations

import numpy as np
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


def test_batch_runs_allocate_no_device_memory():
    grid = 65535  # blocks of a member's scatter, 8 bytes each in the batch's map

    def batch_of(count):
        members = [_solver((16, 12, 12), 20000, seed=i, grid=grid) for i in range(count)]
        return dm.Batch(members)

    warm = batch_of(2)
    warm.set_graphs(False)
    warm.run(3)
    warm.synchronize()
    batch = batch_of(16)
    batch.set_graphs(False)
    before = _free()
    batch.run(3)
    batch.synchronize()
    assert before - _free() < 16 * grid * 8
    batch.close()
    warm.close()


@pytest.mark.parametrize("graphs", [True, False])
def test_batch_follows_scatter_grids(graphs):
    """Smaller and larger maps than the batch was created with."""
    alone = [_solver((24, 12, 12), 30000 + 5000 * i, seed=i) for i in range(3)]
    members = [_solver((24, 12, 12), 30000 + 5000 * i, seed=i) for i in range(3)]
    batch = dm.Batch(members)
    batch.set_graphs(graphs)
    for grid in (None, 3, 5000, 40):
        if grid:
            members[1].set_scatter_grid(grid)
        batch.run(4)
        for a in alone:
            a.DoBenchmark(4, a.settings.dt)
    for a, m in zip(alone, members):
        p, q = a.particles(), m.particles()
        for k in ("pos", "vel", "key"):
            assert np.array_equal(p[k], q[k]), k
        a.close()
    batch.close()
