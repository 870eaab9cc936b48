"""A small problem's step starts and ends in one block each; the launches that
larger problems take instead give the same numbers: the mixed engine's bit for
bit, the FP64 engine's but for the order of its floating-point atomics."""
from __future__ import annotations

import numpy as np
import pytest

from storm_amd import capi
from storm_amd import problems as P
from storm_amd.engine import GpuEngine
from tests.test_gpu_small_steps import SHAPES, make

pytestmark = pytest.mark.gpu

SMALL = [s for s in SHAPES if np.prod(s) <= 2048]


def compare(spec, precision, steps):
    mixed = precision == capi.MIXED
    with GpuEngine(spec, precision) as a, GpuEngine(spec, precision) as b:
        b.general_steps()
        for _ in range(steps):
            a.step()
            b.step()
            ca, cb, ka, kb, La, Lb = a.cells(), b.cells(), a.counters(), b.counters(), a.ledger(), b.ledger()
            for k in ka:
                if not k.startswith("seconds_"):
                    assert ka[k] == kb[k], (k, ka[k], kb[k])
            assert np.array_equal(a.beginning_counts(), b.beginning_counts())
            assert np.array_equal(a.segments(), b.segments())
            ra, rb = a.export_census(), b.export_census()
            assert len(ra) == len(rb) and ra.tobytes() == rb.tobytes()
            if mixed:
                for k in ca:
                    assert np.array_equal(ca[k], cb[k]), k
                assert La == Lb
                ta, tb = a.tallies(), b.tallies()
                for k in ta:
                    assert np.array_equal(ta[k], tb[k]), k
            else:
                # a cell's deposits and path integrals: up to some thousands of positive doubles each, in
                # another order, 1e4 * 2^-53; temperatures and energies are no further off
                for k in ca:
                    assert np.allclose(ca[k], cb[k], rtol=2e-12, atol=0.0), k


@pytest.mark.parametrize("shape", SMALL, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("groups", [0, 4])
@pytest.mark.parametrize("precision", [capi.MIXED, capi.FP64])
def test_routes_agree(shape, groups, precision):
    # the FP64 engine's second step starts from a state that differs in the last bits
    compare(make(shape, groups), precision, 3 if precision == capi.MIXED else 1)


@pytest.mark.parametrize("make_spec", [
    lambda: P.c1_slab(seed=4, packets_scale=0.1, steps=3),
    lambda: P.c3_step(seed=4, nx=32, nyz=4, packets_scale=0.01),
    lambda: P.voronoi_slab(seed=4, n=300, thick=True),
    lambda: P.densmore(nx=64, seed=4, groups=12, new_photons=4, comb_nmin=20)],
    ids=["source", "walk and DDMC", "polyhedra", "groups and walk"])
def test_routes_agree_on_problems(make_spec):
    compare(make_spec(), capi.MIXED, 3)
