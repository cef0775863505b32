"""The packed descriptors of the single-operator calls hold the bytes of their
ctypes structures, and the binding's output extents those of the library."""
import ctypes

import numpy as np
import pytest

from oxionnx_amd import _lib as L
from oxionnx_amd import device as D


def _value(rng, t, i):
    if t is ctypes.c_float:
        return float(np.float32(rng.normal()))
    if issubclass(t, ctypes._Pointer):
        return D._ZERO_POINTS_AT
    return int(rng.integers(-1000, 1000)) + i


@pytest.mark.parametrize("packer", [D._GEMM, D._CONV, D._CONVT, D._MATMUL, D._QGEMM], ids=lambda p: p._desc.__name__)
@pytest.mark.parametrize("beyond_f32", [False, True])
def test_packed_bytes_are_the_structure(packer, beyond_f32):
    desc = packer._desc
    types = [t for _, t in desc._fields_]
    values = [_value(np.random.default_rng(5), t, i) for i, t in enumerate(types)]
    if beyond_f32:
        values = [1e300 if t is ctypes.c_float else v for v, t in zip(values, types)]
    want = desc(*(ctypes.cast(v, t) if issubclass(t, ctypes._Pointer) else v for v, t in zip(values, types)))
    got = desc.from_buffer_copy(packer(*values))
    for (name, t) in desc._fields_:
        a, b = getattr(got, name), getattr(want, name)
        if issubclass(t, ctypes._Pointer):
            a, b = ctypes.addressof(a.contents), ctypes.addressof(b.contents)
        assert a == b, name


@pytest.mark.parametrize("zp", [-128, -1, 0, 127, 128, 255])
def test_zero_point_table(zp):
    assert ctypes.c_int32.from_address(D._ZERO_POINTS_AT + 4 * (zp + 128)).value == zp


def test_output_extents_are_the_library_s():
    rng = np.random.default_rng(6)
    for _ in range(2000):
        v = [int(x) for x in rng.integers(-1, 12, 6)]
        assert D._out_dim(*v) == L.lib().ohip_conv_out_dim(*v), v
