"""The kernels' short forms of reciprocals, reciprocal roots and quotients give
the bits of the division operator and sqrtf: on every float, on each byte by 255,
and in the projection of 2^35 points a seed, of which over a third is in the range
that takes the short form (tests/hip/quotients.hip, which includes the functions)."""
import ctypes as C
import os

import pytest

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "hip", "libquotients.so")


@pytest.fixture(scope="module")
def lib(built):
    import torch  # noqa: F401  (its HIP runtime)
    assert os.path.exists(LIB), "run __graft_entry__.build() first"
    out = C.CDLL(LIB)
    for name in ("check_reciprocal", "check_reciprocal_sqrt", "check_byte", "check_projection"):
        getattr(out, name).restype = C.c_longlong
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["check_reciprocal", "check_reciprocal_sqrt", "check_byte"])
def test_every_value(lib, name):
    first = C.c_uint64()
    bad = getattr(lib, name)(C.byref(first))
    assert bad == 0, "%d values, the first %#x" % (bad, first.value)


@pytest.mark.gpu
@pytest.mark.parametrize("seed", [1, 1 << 40, 1 << 60])
def test_projections(lib, seed):
    first = C.c_uint64()
    bad = lib.check_projection(C.c_uint64(seed), C.c_uint64(1 << 35), C.byref(first))
    assert bad == 0, "%d points, the first %d" % (bad, first.value)
