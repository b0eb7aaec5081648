"""REFERENCE steps whose tiles are taken by single waves, against the oracle:
MT and Hybrid-Taus collision streams, walls, sampling, and tiles too full for
a wave's or the workgroup's LDS (GPU)."""
from __future__ import annotations

import numpy as np
import pytest

import cudadsmc_amd as dm
from cudadsmc_amd import _capi

from helpers import small_reference_settings
from test_gpu_parity import _compare_state, _mirror

pytestmark = pytest.mark.gpu


# at most 200 expected particles in each of 2048 tiles and 300 in each of 4096 go to single waves; the last two are
# the default 64-cell tiles of a large grid. crowd: particles put into the first 32 cells (a wave's LDS holds 496 of
# a tile, the workgroup's 2048)
@pytest.mark.parametrize("dims,ppc,tile,mt,crowd", [
    ((64, 32, 32), 1, 32, 1, 0), ((64, 32, 32), 2, 32, 1, 700), ((64, 32, 32), 6, 32, 0, 0),
    ((64, 64, 32), 2, 32, 0, 2600), ((64, 64, 64), 1, None, 0, 500), ((65, 65, 63), 2, None, 0, 700)])
def test_narrow_reference_tiles_match_oracle(dims, ppc, tile, mt, crowd):
    print(f"narrow REFERENCE tiles dims={dims} ppc={ppc} tile={tile} mt={mt} crowd={crowd}", flush=True)
    s = small_reference_settings(dims=dims, ppc=ppc)
    s.sample_every = 2
    s.mt = mt
    sol = dm.Solver()
    sol.Init(s)
    if tile:
        sol.set_tile_cells(tile)
    assert sol.layout()["tile_cells"] == (tile or 64)
    mesh = dm.icosphere((0.07, 0.06, 0.05), 0.022, 2)
    sol.SetModel(mesh, grid=(6, 6, 6))
    o = _mirror(sol, mesh)
    if not mt:
        o.set_taus(sol.taus_state())
    U = (900.0, 150.0, -120.0)
    n = sol.InitSystemState(U)
    o.load(U)
    assert n == ppc * sol.n_cells
    if crowd:
        p = sol.particles()
        pos, vel = p["pos"].copy(), p["vel"].copy()
        # from anywhere in the box into the first 32 cells, slow enough to stay
        k = np.random.default_rng(crowd).choice(n, crowd, replace=False)
        pos[:, k] *= np.array([[31.5 / dims[0]], [0.96 / dims[1]], [0.96 / dims[2]]], np.float32)
        vel[:, k] *= np.float32(0.02)
        sol.set_particles(pos, vel)
        o.set_state(pos, vel)
    _compare_state(sol, o, "load")
    sol.set_debug(_capi.FLAG_KEEP_PERM | _capi.FLAG_HITS)
    hits = 0
    for step in range(1, 6):
        sol.RunBenchmarkSimulationStep(s.dt)
        o.step(sample=step % 2 == 0)
        start = sol.cell_start()
        assert np.array_equal(start, o.cell_start()), step
        assert crowd == 0 or start[32] > 0.9 * crowd  # still there
        assert np.array_equal(sol.perm(n), o.perm(n)), step
        assert np.array_equal(sol.hit_counts(n), o.hits(n)), step
        hits += int(o.hits(n).sum())
        _compare_state(sol, o, f"step {step}")
        assert np.array_equal(sol.ntc_state(), o.ntc()), step
        if not mt:
            assert np.array_equal(sol.taus_state(), o.taus()), step
    assert np.array_equal(sol.rng_state(), o.rng())
    assert np.array_equal(sol.cell_stats(), o.samples())
    coll, want = sol.collision_stats(), o.cstat().astype(np.float64).sum(0)
    assert np.allclose(coll[:3], want[:3], rtol=1e-12)
    assert hits > 0 and (ppc == 1 or coll[1] > 0)
    sol.close()
