"""A body that cannot be set: no later call's kernel may look at the memory of
the body before it. Runs the engine's host code on a stand-in for the HIP
runtime (host_hip.cpp) in a process of its own."""
from __future__ import annotations

import ctypes as C
import subprocess
import sys
from pathlib import Path

HERE = Path(__file__).resolve().parent


def _child(shim: str) -> None:
    hip = C.CDLL(shim, mode=C.RTLD_GLOBAL)  # before the engine: its calls go to the stand-in
    import cudadsmc_amd as dm
    from helpers import small_physics_settings

    s = small_physics_settings()
    sol = dm.Solver()
    sol.Init(s)
    meshes = [dm.icosphere((0.07, 0.05, 0.05), r, 1) for r in (0.02, 0.01)]
    sol.SetModel(meshes[0], grid=(6, 6, 6))
    whole = sol.fluid_fraction().sum()
    sol.fields()
    assert whole < sol.n_cells and hip.host_hip_launches() > 0 and hip.host_hip_stale() == 0
    failed = 0
    for n in range(40):  # the n-th allocation fails
        hip.host_hip_fail_after(C.c_long(n))
        try:
            sol.SetModel(meshes[1], grid=(6, 6, 6))
        except dm.DsmcError:
            failed += 1
        hip.host_hip_fail_after(C.c_long(-1))
        sol.fields()
        sol.drag()
        assert hip.host_hip_stale() == 0, f"allocation {n}"
    assert 8 <= failed < 40  # every allocation of the body has failed once, and then none
    assert whole < sol.fluid_fraction().sum() < sol.n_cells  # the smaller body at last
    sol.close()
    print("ok", flush=True)


def test_failed_body_leaves_no_freed_memory_in_reach(tmp_path):
    shim = tmp_path / "libhost_hip.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", str(HERE / "host_hip.cpp"), "-o", str(shim)],
                   check=True)
    code = f"import sys; sys.path[:0] = [{str(HERE.parent)!r}, {str(HERE)!r}]; " \
           f"import test_geometry_failure as t; t._child({str(shim)!r})"
    run = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0 and "ok" in run.stdout, run.stdout + run.stderr
