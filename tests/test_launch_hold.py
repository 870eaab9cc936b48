"""Steps that run in a schedule set for them (the no-allocation steps of
multigroup polyhedral problems) leave the schedule watch alone: on the CPU with
made-up rates, and on the GPU past the step where a probe would come."""
from __future__ import annotations

import os
import subprocess

import pytest

from storm_amd import capi
from storm_amd import problems as P

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_watch_ignores_held_steps():
    exe = os.path.join(ROOT, "tests", "cpp", "_build", "launch_hold")
    if not os.path.exists(exe):
        pytest.fail("tests/cpp/_build/launch_hold is not built (run __graft_entry__.build())")
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.count(" ok") == 4, out.stdout


@pytest.mark.gpu
def test_noalloc_steps_keep_the_own_schedule():
    from storm_amd.engine import GpuEngine

    with GpuEngine(P.c4_voronoi(seed=15, n=500, groups=8, packets_scale=0.005), capi.MIXED) as e:
        for _ in range(40):
            e.step_noalloc()
            assert e.counters()["transport_schedule"] == capi.SCHEDULE_PASS
            assert e.launch()["schedule"] == capi.SCHEDULE_REFILL
        e.step()
        assert e.counters()["transport_schedule"] == capi.SCHEDULE_REFILL
