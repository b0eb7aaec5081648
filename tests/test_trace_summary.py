"""The kernel-trace summariser finds the steps of either scan form (CPU)."""
from __future__ import annotations

import csv
import sys

import pytest

from cudadsmc_amd import trace_summary


@pytest.mark.parametrize("scan", [["k_scan_small(x)"], ["k_scan_reduce_step(x)", "k_scan_apply_step(x)"]])
def test_steps_are_found(tmp_path, monkeypatch, capsys, scan):
    path, t = tmp_path / "run_kernel_trace.csv", 0
    with open(path, "w", newline="") as f:
        w = csv.writer(f)
        w.writerow(["Kernel_Name", "Start_Timestamp", "End_Timestamp", "Grid_Size_X", "Grid_Size_Y"])
        for step in range(6):
            for name in [*scan, "k_scatter(x)", "void k_tile<1u, false>(x)", "k_walls(x)"]:
                w.writerow([name, t, t + 1000 * (step + 1), 262144, 1])
                t += 10000
    monkeypatch.setattr(sys, "argv", ["trace_summary", str(path), "--skip", "1", "--take", "3"])
    trace_summary.main()
    out = capsys.readouterr().out
    assert "main-workload steps in trace: 6; summarised: steps 2-4" in out
    assert "| `k_tile<1u, false>` | 1.00 | 3.0 | 3.0 |" in out
