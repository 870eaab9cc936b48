"""Gray cells without absorption in the mixed engine: their path integral goes
where other cells' deposit goes, is the replay's bit for bit, and costs what a
deposit costs."""
from __future__ import annotations

import numpy as np
import pytest

from storm_amd import capi
from storm_amd import problems as P
from storm_amd.engine import GpuEngine

pytestmark = pytest.mark.gpu


def line(cells, sigma_a, sigma_s, scale=1.0, accel=False):
    """A 1 cm line of cells that do not absorb (and so emit nothing) but where sigma_a says."""
    spec = P.c1_slab(seed=7, nx=cells, packets_scale=scale, steps=2)
    spec.sigma_a0 = np.broadcast_to(np.asarray(sigma_a, dtype=np.float64), cells).copy()
    spec.sigma_s0 = np.full(cells, float(sigma_s))
    if accel:
        spec.with_rw = spec.with_ddmc = 1
        spec.rw_cell_tau = spec.ddmc_cell_tau = spec.rw_particle_tau = 10.0
    return spec


def every_other(cells):
    s = np.zeros(cells)
    s[::2] = 2.0
    return s


# 1 to 2048 cells end their step in one block, more in kernels of their own
@pytest.mark.parametrize("cells,absorbing,sigma_s,accel", [
    (1, False, 3.0, False), (37, True, 3.0, False), (37, False, 0.0, False), (2100, True, 30.0, False),
    (60, True, 2000.0, True)])
def test_path_integral_is_the_replays(oracle, cells, absorbing, sigma_s, accel):
    spec = line(cells, every_other(cells) if absorbing else 0.0, sigma_s, scale=0.2, accel=accel)
    with GpuEngine(spec, capi.MIXED) as e:
        e.step()
        e.keep_transport_inputs(True)
        e.step()
        pk, n, xs, consts = e.transport_inputs()
        got, c, counts = e.tallies(), e.cells(), e.counters()
        ref, out = oracle.replay_transport(spec, pk, n, xs, consts, accel=e.accel_data())
    assert n > 0 and (counts["random_walk_steps"] > 0) == accel
    for k in ("segs", "dep", "rdep", "pint", "esc"):
        assert np.array_equal(got[k].astype(np.uint64), ref[k].astype(np.uint64)), k
    absorbs = xs[0::2] > 0
    dep, pint = got["dep"][0::2], got["pint"][0::2]
    assert not dep[~absorbs].any() and not pint[absorbs].any()
    assert pint[~absorbs].any() and dep[absorbs].any() == absorbs.any()
    # erad = path integral / (c dt V): the conversion from integers and a quotient, in doubles
    want = pint[~absorbs].astype(np.float64) * 2.0 ** consts[3] / (P.CLIGHT * spec.dt * spec.volumes()[~absorbs])
    assert np.allclose(c["erad"][~absorbs], want, rtol=1e-14, atol=0.0)


def test_polyhedral_cells():
    spec = line(64, every_other(64), 3.0, scale=0.2)
    spec.umesh = P.cartesian_umesh(spec.x_edges, spec.y_edges, spec.z_edges)
    with GpuEngine(spec, capi.MIXED) as e:
        e.step()
        t, L = e.tallies(), e.ledger()
    absorbs = spec.sigma_a0 > 0
    dep, pint = t["dep"][0::2], t["pint"][0::2]
    assert not dep[~absorbs].any() and not pint[absorbs].any() and dep[absorbs].any() and pint[~absorbs].any()
    assert L["census_in"] + L["emitted"] + L["source"] == L["deposited"] + L["escaped"] + L["census_pre"]


def test_cost_is_a_deposits():
    """A slab that only scatters against one that also absorbs a millionth per cm: the same histories and
    one tally a visit in both.  1.5: with the path integral in one word a cell for the whole device the
    ratio is above 3, shared words leave it near 1."""
    ms = []
    for sigma_a in (0.0, 1e-6):
        with GpuEngine(line(100, sigma_a, 100.0, scale=10.0), capi.MIXED) as e:
            e.set_tuning(block=256, schedule=capi.SCHEDULE_REFILL)
            t = []
            for _ in range(6):
                e.step()
                t.append(e.counters()["seconds_transport"] * 1e3)
            ms.append(min(t[2:]))
    print("transport, ms a step: only scattering %.3f, with absorption %.3f" % tuple(ms))
    assert ms[0] <= 1.5 * ms[1], ms
