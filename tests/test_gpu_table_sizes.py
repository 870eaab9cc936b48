"""The block's LDS tally table is sized by its range of packets, the mesh's
cells and the LDS a block has: results do not depend on it, from one cell to
meshes that no table holds, in every block size."""
from __future__ import annotations

import numpy as np
import pytest

from storm_amd import capi
from storm_amd import problems as P
from storm_amd.engine import GpuEngine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [1, 511, 513, 900, 4096])
@pytest.mark.parametrize("block", [64, 128, 256, 512])
@pytest.mark.parametrize("precision", [capi.MIXED, capi.FP64])
def test_results_do_not_depend_on_the_table(cells, block, precision):
    spec = P.c1_slab(seed=2, nx=cells, packets_scale=20.0 / max(cells, 20), steps=1)
    out = []
    # a range of 64 packets a wavefront, whose table the cells decide, and one of 1024, cut to what fills the device
    for chunks, schedule in ((1, capi.SCHEDULE_REFILL), (1, capi.SCHEDULE_PASS), (16, capi.SCHEDULE_REFILL)):
        with GpuEngine(spec, precision) as e:
            e.set_tuning(block=block, schedule=schedule)
            e.set_chunks_per_wave(chunks)
            e.step()
            out.append((e.segments(), e.cells(), e.counters()["segments"], e.export_census()))
    seg, c, n, rec = out[0]
    assert n > 0 and int(seg.sum()) == n
    for s, d, m, r in out[1:]:
        assert m == n and np.array_equal(s, seg) and len(r) == len(rec)
        for k in c:
            if precision == capi.MIXED:
                assert np.array_equal(c[k], d[k]), k
            else:  # up to some 1e4 positive doubles a cell in another order, 1e4 * 2^-53
                assert np.allclose(c[k], d[k], rtol=2e-12, atol=0.0), k
