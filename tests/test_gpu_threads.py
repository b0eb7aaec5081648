"""Handles of several host threads: a read waits for its own handle's steps,
not for those of another (GPU)."""
from __future__ import annotations

import threading
import time

import numpy as np
import pytest

import cudadsmc_amd as dm

from helpers import small_physics_settings

pytestmark = pytest.mark.gpu


def _solver(dims, n, seed=1):
    s = small_physics_settings(dims=dims, n_target=n)
    s.seed = seed
    sol = dm.Solver()
    sol.Init(s)
    sol.InitSystemState(tuple(s.stream_velocity))
    return sol


def test_reads_of_one_handle_do_not_wait_for_another():
    busy = _solver((64, 64, 64), 4000000)
    others = [_solver((64, 64, 32), 200000, seed=2 + i) for i in range(4)]  # fields of more than one half-buffer
    for sol in [busy] + others:  # every kernel and buffer of the calls below has been used once
        sol.set_sampling(True)
        sol.DoBenchmark(5, sol.settings.dt)
        sol.drag()
        sol.fields()
    for _ in range(3):  # the last one from steps captured before
        t0 = time.perf_counter()
        busy.DoBenchmark(101, busy.settings.dt)
        busy.synchronize()
    steps = int(np.clip(101 * 1.5 / (time.perf_counter() - t0), 100, 20000))  # about 1.5 s of them
    order, fields = [], {}

    def read(name, sol):
        sol.drag()
        fields[name] = sol.fields()
        order.append((name, round(time.perf_counter() - t0, 3)))

    t0 = time.perf_counter()
    busy.DoBenchmark(steps, busy.settings.dt)
    print(f"{steps} steps queued in {time.perf_counter() - t0:.3f} s", flush=True)
    first = threading.Thread(target=read, args=("busy", busy))
    first.start()
    time.sleep(0.1)  # its read is waiting for the steps now
    threads = [threading.Thread(target=read, args=(i, sol)) for i, sol in enumerate(others)]
    for t in threads:
        t.start()
    for t in threads + [first]:
        t.join()
    print(f"reads ended at {order}", flush=True)
    # streams share the GPU's few hardware queues, so some of the four may have
    # to wait behind the steps; one that has a queue of its own does not
    assert order[0][0] != "busy"
    for name, sol in [("busy", busy)] + list(enumerate(others)):
        again = sol.fields()
        assert np.any(again["T"] > 0.0)
        for k, v in again.items():
            np.testing.assert_array_equal(fields[name][k], v, err_msg=k)
        sol.close()
