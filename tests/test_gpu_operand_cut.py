"""The cut of fp32 operands into three bf16 parts loses nothing: every significand times 1, in either half of a pair."""
import ctypes

import numpy as np
import pytest

from alpha2_amd import _ffi as ffi
from alpha2_amd.backend import TensorData

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def B():
    from alpha2_amd import HipBackend
    return HipBackend(0)


# exponents of the two halves, beside each other and far apart, to both ends of what the cut takes (2^104 on is the fp32 instruction's)
@pytest.mark.parametrize("low,high", [(0, 0), (0, -1), (-126, -126), (-126, 103), (103, 103), (60, -30), (-8, 7), (1, -24)])
@pytest.mark.parametrize("rows,n,kernel", [(1024, 256, b"pieces"), (1 << 17, 64, b"split")])
def test_every_significand_times_one(B, rows, n, kernel, low, high):
    """A product with the identity: a result is the sum of its value's three parts (the other terms are zeros), which is exact if the
    parts are what the cut says they are."""
    bits = np.arange(1 << 23, dtype=np.uint32).reshape(-1, n)
    a = (bits | np.uint32(0x3F800000)).view(np.float32)
    a[1::2] *= -1
    a[:, 0::2] = np.ldexp(a[:, 0::2], low)
    a[:, 1::2] = np.ldexp(a[:, 1::2], high)
    one, name = TensorData((n, n), "f32", np.eye(n, dtype=np.float32)), ctypes.create_string_buffer(200)
    for part in np.split(a, a.shape[0] // rows):
        got = B.matmulTransposed(TensorData(part.shape, "f32", part), one)
        ffi.check(B.lib.ah_gemm_last_kernel(name, 200, None))
        assert kernel in name.value, name.value
        assert np.array_equal(got.data.view(np.uint32), part.reshape(-1).view(np.uint32))
