"""Dropout masks where the hash leaves whole-number arithmetic: around the index from which the sum passes 2^53, which comes earlier for
higher mask numbers and at once for the highest, against doubles."""
import numpy as np
import pytest

from alpha2_amd import _ffi as ffi

pytestmark = pytest.mark.gpu
MUL = 2246822519


@pytest.fixture(scope="module")
def B():
    from alpha2_amd import HipBackend
    return HipBackend(0)


def _mask(seed, counter, p, n):
    s = (float(seed) + float(counter) * 2654435761.0) + np.arange(n, dtype=np.float64) * float(MUL)
    h = (s.astype(np.int64) & 0xffffffff).astype(np.uint64)
    h = ((h ^ (h >> np.uint64(16))) * np.uint64(0x85ebca6b)) & np.uint64(0xffffffff)
    h = ((h ^ (h >> np.uint64(13))) * np.uint64(0xc2b2ae35)) & np.uint64(0xffffffff)
    h = h ^ (h >> np.uint64(16))
    return np.where(h.astype(np.float64) * (1.0 / 4294967296.0) > p, np.float32(1.0 / (1.0 - p)), np.float32(0))


def _whole(counter):
    return max(0, int((2.0 ** 53 - 2.0 ** 31 - abs(counter) * 2654435761.0) / MUL))


@pytest.mark.parametrize("counter", [0, 15, -15, 3_000_000, 3_393_200, -3_393_200, 2 ** 31 - 1, -2 ** 31])
@pytest.mark.parametrize("seed,p", [(42, 0.1), (-2 ** 31, 0.0), (2 ** 31 - 1, 0.999)])
def test_masks_on_both_sides(B, counter, seed, p):
    n = _whole(counter) + 1003
    want = _mask(seed, counter, p, n)
    assert np.array_equal(B.dropoutMask([n], seed, counter, p).data, want)
    x, s = B.full([n], 1.0), B.fromArray([seed], [1], "i32")
    for residual in (0, B._ptr(x)):
        for shift in (0, 1):                        # four elements a thread, and one
            out = B._new([n])
            ffi.check(B.lib.ah_dropout_apply(B._ptr(x) + 4 * shift, ffi.F32, residual + 4 * shift if residual else 0, out._buf.ptr + 4 * shift, ffi.F32, n - shift,
                                             B._ptr(s), counter, p))
            got = out.data[shift:]
            assert np.array_equal(got, want[:n - shift] + np.float32(1 if residual else 0))
