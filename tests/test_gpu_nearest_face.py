"""The polyhedral tracker's two ways to the nearest face: with short divisions
on a mesh whose planes all lie 2^-30 to 2^50 cm from their cell's mesh point,
with IEEE divisions on any other."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from storm_amd import capi
from storm_amd import problems as P
from storm_amd.engine import GpuEngine

pytestmark = pytest.mark.gpu


def with_island(spec, offset):
    """`spec` and, as its last cell, a cube of its own that no packet enters
    or leaves, its mesh point `offset` cm from one of its faces."""
    m, h = spec.umesh, 0.1
    edges = np.array([0.0, h])
    c = P.cartesian_umesh(edges, edges, edges)
    nbr = np.full(6, -3, dtype=np.int32)  # reflecting box side
    point = c.mesh_point.copy()
    point[0, 0] = offset
    spec.umesh = P.UMesh(
        volume=np.concatenate([m.volume, c.volume]), mesh_point=np.concatenate([m.mesh_point, point]),
        face_start=np.concatenate([m.face_start, [m.nfaces + 6]]).astype(np.uint32),
        face_neighbor=np.concatenate([m.face_neighbor, nbr]).astype(np.int32),
        face_normal=np.concatenate([m.face_normal, c.face_normal]),
        face_centroid=np.concatenate([m.face_centroid, c.face_centroid]),
        face_area=np.concatenate([m.face_area, c.face_area]),
        face_vertex_start=np.concatenate([m.face_vertex_start, c.face_vertex_start[1:] + m.face_vertex_start[-1]])
        .astype(np.uint32),
        vertices=np.concatenate([m.vertices, c.vertices]), box_lo=m.box_lo, box_hi=m.box_hi)
    for k in ("sigma_a0", "sigma_s0", "T0", "density"):
        v = getattr(spec, k)
        if v is not None:
            setattr(spec, k, np.concatenate([v, v[:1]]))
    return spec


@pytest.mark.parametrize("thick,groups", [(False, 0), (True, 0), (False, 8)])
@pytest.mark.parametrize("offset", [1e-10, 1e-30])
def test_general_meshes_give_the_same_bits(thick, groups, offset):
    """An island whose mesh point lies next to a face puts the whole mesh on the general path; the
    other cells' first step is then that of the short one, bit for bit."""
    out = []
    for x in (0.05, offset):
        spec = with_island(P.voronoi_slab(seed=5, n=300, thick=thick, groups=groups), x)
        with GpuEngine(spec, capi.MIXED) as e:
            e.step()
            L = e.ledger()
            assert L["census_in"] + L["emitted"] + L["source"] == L["deposited"] + L["escaped"] + L["census_pre"]
            assert int(e.segments()[-1]) > 0
            out.append((e.cells(), e.tallies(), e.segments()))
    (ca, ta, sa), (cb, tb, sb) = out
    assert sa[:-1].sum() > 10000 and np.array_equal(sa[:-1], sb[:-1])
    for k in ca:
        assert np.array_equal(ca[k][:-1], cb[k][:-1]), k
    for k in ("dep", "pint", "rdep", "esc"):
        assert np.array_equal(ta[k][:-2], tb[k][:-2]), k


@pytest.mark.parametrize("first,count", [(0, 1), (0, 257), (1, 1 << 22)])
def test_median_passes_over_no_number(first, count):
    """A quotient that is no number (a denominator too small for the short division) leaves the smaller
    distance as the second, which sends the segment to the exact search."""
    lib = capi.load_library()
    bad = C.c_uint64()
    assert lib.storm_gpu_debug_math(5, first, count, C.byref(bad)) == 0, lib.storm_gpu_last_error()
    assert bad.value == 0
