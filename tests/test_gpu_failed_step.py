"""The per-cell counts and tallies after a step that stopped part-way: this
step's, in problems of the one-block route (up to 2048 cells) and beyond."""
from __future__ import annotations

import numpy as np
import pytest

from storm_amd import capi
from storm_amd import problems as P
from storm_amd.engine import GpuEngine, StormError

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [100, 2100])
def test_census_that_outgrows_its_buffer(cells):
    """Without population control the census grows until a no-allocation step has no room for it, which
    is found after the transport: the segments and deposits are those of the same step with allocations."""
    spec = P.c1_slab(seed=9, nx=cells, packets_scale=30.0 / cells, steps=200)
    spec.comb = 0
    with GpuEngine(spec, capi.MIXED) as ref, GpuEngine(spec, capi.MIXED) as e:
        for _ in range(spec.steps):
            ref.step()
            try:
                e.step_noalloc()
            except StormError as err:
                assert "must grow" in str(err), err
                break
        else:
            pytest.fail("no step was refused")
        assert ref.counters()["segments"] > 0
        assert np.array_equal(e.segments(), ref.segments())
        assert np.array_equal(e.beginning_counts(), ref.beginning_counts())
        a, b = e.tallies(), ref.tallies()
        for k in ("dep", "pint", "rdep", "esc", "segs"):
            assert np.array_equal(a[k], b[k]), k


@pytest.mark.parametrize("cells", [100, 2100])
def test_step_refused_before_the_transport(cells):
    spec = P.c1_slab(seed=9, nx=cells, packets_scale=4000.0 / cells, steps=2)
    with GpuEngine(spec, capi.MIXED) as e:
        e.step()
        assert e.segments().any()
        with pytest.raises(StormError, match="error 4"):
            e.step_noalloc()
        assert not e.segments().any() and not e.tallies()["dep"].any()
