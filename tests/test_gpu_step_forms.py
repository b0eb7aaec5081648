"""The forms that a step takes by the size of an instance: the scan of one or
two launches at its limits, several blocks of freestream faces, the wall pass
from the bitmask or from the compacted list (GPU)."""
from __future__ import annotations

import numpy as np
import pytest

import cudadsmc_amd as dm

from helpers import small_physics_settings
from test_gpu_batch import make
from test_gpu_parity import _compare_state, _mirror

pytestmark = pytest.mark.gpu


# cells: one block of 4096; not a multiple of four; the most of the one-launch scan (16 blocks, 10240 faces in three
# blocks); two launches with an odd rest; a long thin box with more faces than cells; the second and the fourth with
# tile queues, whose cells' counts come from two arrays; one tile of 16 cells with about 94 particles each
@pytest.mark.parametrize("dims,n", [((16, 16, 16), 20000), ((17, 13, 19), 9000), ((64, 32, 32), 40000),
                                    ((65, 33, 31), 40000), ((5000, 1, 1), 20000),
                                    ((17, 13, 19), 60000), ((65, 33, 31), 600000), ((4, 2, 2), 1500)])
def test_step_forms_match_oracle(dims, n):
    print(f"step forms dims={dims} n={n}", flush=True)
    s = small_physics_settings(dims=dims, n_target=n)
    sol = dm.Solver()
    sol.Init(s)
    mesh = dm.icosphere((0.07, 0.05, 0.05), 0.02, 2)
    sol.SetModel(mesh, grid=(6, 6, 6))
    o = _mirror(sol, mesh)
    sol.InitSystemState((1500.0, 0.0, 0.0))
    o.load((1500.0, 0.0, 0.0))
    for k in range(5):
        sol.RunBenchmarkSimulationStep(s.dt)
        o.step(sample=False)
        assert np.array_equal(sol.cell_start(), o.cell_start()), k
        _compare_state(sol, o, f"step {k + 1}")
    assert np.array_equal(sol.ntc_state(), o.ntc())
    sol.close()


def test_wall_forms_give_the_same_walls():
    """Members of a batch that is large as a whole take the list, the same
    solvers on their own the bitmask: state and wall sums agree, also where
    the forms alternate and the host reads the sums in between."""
    args = [(1 + i, 100000 + 1000 * i, 900.0 + 100.0 * i, 0.015 + 0.001 * i) for i in range(12)]
    alone = [make(*a) for a in args]
    members = [make(*a) for a in args]
    batch = dm.Batch(members)
    for steps in (3, 2):
        for a, m in zip(alone, members):
            a.DoBenchmark(steps + 1, a.settings.dt)
        batch.run(steps)
        for i, m in enumerate(members):
            m.RunBenchmarkSimulationStep(m.settings.dt)  # from the bitmask, after the list
            if i % 3 == 0:
                m.drag()
    for a, m in zip(alone, members):
        p, q = a.particles(), m.particles()
        for k in ("pos", "vel", "key"):
            assert np.array_equal(p[k], q[k]), k
        assert np.any(a.drag() != 0.0) and np.array_equal(a.drag(), m.drag())
        assert np.array_equal(m.drag(), m.drag())  # a second read folds nothing twice
        a.close()
    batch.close()


@pytest.mark.parametrize("mode", [dm.MODE_PHYSICS, dm.MODE_REFERENCE])
def test_fields_from_the_sums(mode):
    """Fields computed on the GPU against the same formulas on the sums, both
    read through the staging halves (several rounds of them in PHYSICS)."""
    if mode == dm.MODE_PHYSICS:
        s = small_physics_settings(dims=(128, 64, 32), n_target=60000)
        steps, kb = 3, 1.380649e-23
    else:
        from helpers import small_reference_settings

        s = small_reference_settings(geometry=False)
        s.sample_every = 2
        steps, kb = 4, float(np.float32(1.3806e-23))
    sol = dm.Solver()
    sol.Init(s)
    if mode == dm.MODE_PHYSICS:
        sol.SetModel(dm.icosphere((0.07, 0.05, 0.05), 0.02, 2), grid=(6, 6, 6))
        frac = sol.fluid_fraction().astype(np.float64)
    else:
        frac = 1.0
    sol.InitSystemState(tuple(s.stream_velocity))
    sol.set_sampling(True)
    sol.DoBenchmark(steps, s.dt)
    samples = sol.counts()[2]
    N, sx, sy, sz, s2 = sol.cell_stats().T
    d = sol.derived()
    vol = float(d["cell_volume"]) * frac
    safe, on = np.maximum(N, 1.0), N > 0
    want = {"n": np.where(vol > 0, float(d["fnum"]) * N / np.where(vol > 0, vol * samples, 1.0), 0.0)}
    u = {k: np.where(on, a / safe, 0.0) for k, a in (("u", sx), ("v", sy), ("w", sz))}
    want.update(u)
    T = float(np.float32(s.molmass)) * (s2 / safe - (u["u"] ** 2 + u["v"] ** 2 + u["w"] ** 2)) / (3.0 * kb)
    want["T"] = np.where(on, T, 0.0)
    assert samples > 0 and on.any()
    got = sol.fields()
    for k, w in want.items():
        np.testing.assert_array_equal(got[k], w.astype(np.float32), err_msg=k)
    sol.close()


def _narrow_pair(tile_cells, crowd, seed=11, dims=(64, 64, 32), n=60000):
    """Two equal solvers, tiles of `tile_cells` (taken by single waves) and of
    128 cells (by workgroups). `crowd` of the particles are put into the first
    32 cells: more than a wave's share of the LDS, or than all of it."""
    out = []
    for tc in (tile_cells, 128):
        s = small_physics_settings(dims=dims, n_target=n)
        s.seed = seed
        sol = dm.Solver()
        sol.Init(s)
        sol.set_tile_cells(tc)
        sol.SetModel(dm.icosphere((0.07, 0.05, 0.05), 0.02, 2), grid=(8, 8, 8))
        sol.InitSystemState((1500.0, 0.0, 0.0))
        if crowd:
            p = sol.particles()
            pos, vel = p["pos"].copy(), p["vel"].copy()
            k = np.random.default_rng(seed).choice(pos.shape[1], crowd, replace=False)
            pos[:, k] *= np.array([[0.48], [0.96 / dims[1]], [0.96 / dims[2]]], np.float32)
            vel[:, k] *= np.float32(0.02)
            sol.set_particles(pos, vel)
        out.append(sol)
    return out


def _assert_same_run(a, b):
    p, q = a.particles(), b.particles()
    for k in ("pos", "vel", "key"):
        assert np.array_equal(p[k], q[k]), k
    assert np.array_equal(a.ntc_state(), b.ntc_state())
    assert np.array_equal(a.cell_stats(), b.cell_stats())
    assert np.array_equal(a.collision_stats(), b.collision_stats())
    assert np.array_equal(a.drag(), b.drag())


@pytest.mark.parametrize("tile_cells", [32, 64])
@pytest.mark.parametrize("crowd", [0, 497, 1500, 5000])
def test_narrow_tiles_match_wide_tiles(tile_cells, crowd):
    print(f"narrow tiles of {tile_cells} cells, crowd {crowd}", flush=True)
    a, b = _narrow_pair(tile_cells, crowd)
    for sol in (a, b):
        sol.set_sampling(True)
        sol.DoBenchmark(4, sol.settings.dt)
    start = a.cell_start()
    assert crowd == 0 or start[32] > 0.9 * crowd  # still crowded after the steps
    _assert_same_run(a, b)
    a.close()
    b.close()


@pytest.mark.parametrize("members", [1, 3])  # 4096 tiles: one per wave; 12288: a wave walks over four
def test_narrow_tiles_in_a_batch(members):
    pairs = [_narrow_pair(32, 900 * i, seed=5 + i) for i in range(members)]
    extra = _narrow_pair(256, 0, seed=3, dims=(16, 12, 11), n=40000)  # a member taken by workgroups
    batch = dm.Batch([p[0] for p in pairs] + [extra[0]])
    batch.set_sampling(True)
    batch.run(4)
    batch.synchronize()
    for a, b in pairs + [extra]:
        b.set_sampling(True)
        b.DoBenchmark(4, b.settings.dt)
        _assert_same_run(a, b)
        b.close()
    batch.close()


# 128-cell tiles would be 8000: 1024 workgroups; 256-cell tiles 32768: 4096
@pytest.mark.parametrize("dims,n,streams", [((160, 80, 80), 4000000, 1024 * 256), ((512, 128, 128), 8000000, 4096 * 256)])
def test_narrow_tiles_keep_the_streams(dims, n, streams):
    """The random-number streams, and so the particles that a case loads, do
    not go by the size of tiles that single waves take."""
    s = small_physics_settings(dims=dims, n_target=n)
    s.n_streams = 0
    sol = dm.Solver()
    sol.Init(s)
    layout = sol.layout()
    assert layout["tile_cells"] == 64 and layout["n_streams"] == streams
    sol.close()
