"""The mixed engine's short arithmetic forms (storm_amd/csrc/common/fpmath.h)
give the same bits as what they stand for: the correctly rounded reciprocal,
square root and quotient, and the full logarithm and expm1.  Every test is for
equal bits, so there is no tolerance to choose."""
import ctypes as C

import numpy as np
import pytest

from storm_amd import capi


def bits(x):
    return int(np.float32(x).view(np.uint32))


def host(oracle_lib, which, x):
    x = np.ascontiguousarray(x, dtype=np.float32)
    y = np.empty_like(x)
    fp = C.POINTER(C.c_float)
    oracle_lib.replay_fpmath.argtypes = [C.c_int32, C.c_int64, fp, fp]
    oracle_lib.replay_fpmath(which, len(x), x.ctypes.data_as(fp), y.ctypes.data_as(fp))
    return y.view(np.uint32)


# (function, its short form): every value of a uniform, and 1 minus it; for
# expm1 every exponent, dense about the joint of its two series
@pytest.mark.parametrize("full,short,kind", [(0, 5, "uniform"), (0, 5, "rest"), (2, 6, "all"), (2, 6, "joint")])
def test_host_forms_have_the_same_bits(oracle, full, short, kind):
    lib = oracle.rlib()
    if kind in ("uniform", "rest"):
        k = np.arange(1 << 24, dtype=np.float64)[::7]
        u = ((k.astype(np.float32) + np.float32(0.5)) * np.float32(2.0 ** -24)).astype(np.float32)
        x = u if kind == "uniform" else np.float32(1.0) - u
        x = x[x > 0]
    elif kind == "all":
        b = np.arange(0x80000000, 0xFF800000, 997, dtype=np.uint64).astype(np.uint32)  # -0 .. below -inf
        x = b.view(np.float32)
    else:
        j = bits(np.float32(-0.34657359))
        x = np.arange(j - 200000, j + 200000, dtype=np.uint32).view(np.float32)
    assert np.array_equal(host(lib, full, x), host(lib, short, x))


def span(lo, hi):
    return bits(lo), bits(hi) - bits(lo)


@pytest.mark.gpu
@pytest.mark.parametrize("op,ranges", [
    (0, [span(2.0 ** -126, 2.0 ** 126), span(-(2.0 ** -126), -(2.0 ** 126))]),
    (1, [(0, 1), span(2.0 ** -100, 2.0 ** 100)]),
    (2, [span(2.0 ** -25, 1.0), (bits(1.0), 1)]),
    (3, [(0x80000000, 0x7F800000)]),
    (4, [(0, 1 << 28)]),
], ids=["reciprocal", "sqrt", "log", "expm1", "quotient"])
def test_device_forms_have_the_same_bits(op, ranges):
    lib = capi.load_library()
    for first, count in ranges:
        bad = C.c_uint64()
        assert lib.storm_gpu_debug_math(op, first, count, C.byref(bad)) == 0, lib.storm_gpu_last_error()
        assert bad.value == 0, (op, hex(first), count, bad.value)
