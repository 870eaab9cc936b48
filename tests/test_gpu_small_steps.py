"""Steps whose start and end run as one block each (up to 2048 cells and 4096
Z-order codes) and steps on either side of that line.

Both routes have to give the same numbers: the photon allocation worked out
here from the opacities the transport was given, its packets where it puts
them, segments and census that add up, and a ledger that closes exactly.
"""
from __future__ import annotations

import numpy as np
import pytest

from storm_amd import capi
from storm_amd import problems as P
from storm_amd.engine import GpuEngine

pytestmark = pytest.mark.gpu

N_MIN = 7
# cells: 1, a wavefront less one, a block, one more, the limit, one more; 729 cells with the most codes, 1377 with
# more; a cube, lines and slabs beyond
SHAPES = [(1, 1, 1), (63, 1, 1), (1024, 1, 1), (1025, 1, 1), (2048, 1, 1), (2049, 1, 1), (9, 9, 9), (17, 9, 9),
          (4096, 1, 1), (241, 17, 1), (16, 16, 16), (3, 5, 7),
          (65, 9, 3), (33, 17, 5)]


def make(shape, groups=0):
    n = int(np.prod(shape))
    rng = np.random.default_rng(n)
    T0 = P.KEV_K * (0.2 + rng.random(n))
    T0[rng.random(n) < 0.1] = 1e-3 * P.KEV_K if n > 8 else P.KEV_K  # cold cells
    edges = [np.linspace(0.0, 0.01 * k, k + 1) for k in shape]
    kw = dict(group_bounds=np.geomspace(1e-2, 30.0, groups + 1) * P.KEV, nu_pow=3.0, nu_ref=P.KEV) if groups else {}
    return P.ProblemSpec(
        name="small_step", x_edges=edges[0], y_edges=edges[1], z_edges=edges[2],
        sigma_a0=1.0 + 20.0 * rng.random(n), T0=T0, dt=1e-11, steps=2,
        eos_f=1e15 / P.KEV_K, eos_beta=1.0, eos_mu=0.0, face_kind=(capi.FACE_ESCAPE,) * 6,
        source_face=-1, source_T=P.KEV_K, freeze_T4=0, source_per_face=0, new_photons_per_cell=N_MIN,
        comb=1, comb_nmin=5, comb_factor=1.0, seed=3, **kw)


def expected_counts(spec, sig_abs):
    """(lowest, highest) photons per cell; the opacities are known to 2^-24."""
    # emission energy: f V a T^4 sigma dt c, and f sigma is the transport's sig_abs
    E = sig_abs.astype(np.float64) * spec.volumes() * spec.T0 ** 4
    share = E / E.sum() * (spec.ncells * N_MIN * 10)
    eps = 2.0 ** -22  # own rounding and that of the sum, 2^-24 each, and a margin
    return [np.where(E > 0, np.clip(np.floor(share * (1 + s * eps)), N_MIN, 20 * N_MIN), 0) for s in (-1, 1)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("groups", [0, 4])
@pytest.mark.parametrize("precision", [capi.MIXED, capi.FP64])
def test_step_of_a_small_problem(shape, groups, precision):
    spec = make(shape, groups)
    mixed = precision == capi.MIXED
    with GpuEngine(spec, precision) as e:
        for step in range(spec.steps):
            if mixed:
                e.keep_transport_inputs(step == 0)
            e.step()
            c, L = e.counters(), e.ledger()
            begin = e.beginning_counts()
            assert int(begin.sum()) == c["start_particles"] == c["emitted_particles"] + c["initial_particles"]
            if step == 0 and mixed and not groups:
                xs = e.transport_inputs()[2]
                lo, hi = expected_counts(spec, xs[0::2])
                assert ((lo <= begin) & (begin <= hi)).all(), (lo, begin, hi)
            assert int(e.segments().astype(np.int64).sum()) == c["segments"]
            rec, cells = e.export_census(), e.cells()
            assert len(rec) == c["end_particles"]
            if mixed:
                assert L["census_in"] + L["emitted"] + L["source"] == L["deposited"] + L["escaped"] + L["census_pre"]
                assert L["census_pre"] == L["census_out"] + L["comb_rem"] + L["comb_dropped"]
                # an integer of quanta below 2^62 held in a double per cell
                w = float(L["census_out"]) * 2.0 ** L["eq"]
                assert abs(cells["census"].sum() - w) <= 1e-12 * w
            dmat = L["material_after"] - L["material_before"]
            Q = 2.0 ** L["eq"]
            expect = (float(L["deposited"]) - float(L["emitted"]) + float(L["comb_rem"])) * Q + L["requant_rem"] + L["clamp"]
            scale = L["material_before"] + float(L["census_in"] + L["emitted"] + L["source"]) * Q
            assert abs(dmat - expect) <= 1e-12 * scale, (dmat, expect, scale)


def test_small_step_batch_keeps_the_general_path():
    """One instance as a batch (never the one-block route) against the same
    problem by itself: same photons, and a closed ledger on both."""
    d = dict(P.c5_instances(count=1, seed=5, packets_scale=0.02)[0])
    with GpuEngine(P.c5_batch([d], seed=5, steps=1), capi.MIXED) as a, \
            GpuEngine(P.c5_instance_spec(d, seed=5, steps=1), capi.MIXED) as b:
        a.step()
        b.step()
        for e in (a, b):
            L = e.ledger()
            assert L["census_in"] + L["emitted"] + L["source"] == L["deposited"] + L["escaped"] + L["census_pre"]
        assert a.counters()["emitted_particles"] == b.counters()["emitted_particles"]
