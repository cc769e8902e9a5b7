"""gelu and its backward from an fp32 product whose contraction is cut into slices: the kernel that joins them computes both, with the bits of
the calls it stands for; in one piece where slices gain too little for a second launch, and on the side stream."""
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


def _draw(seed, *shape):
    return TensorData(shape, "f32", np.random.default_rng(seed).standard_normal(shape, dtype=np.float32))


def _slices(B):
    name, n = ctypes.create_string_buffer(200), ctypes.c_int32()
    ffi.check(B.lib.ah_gemm_last_kernel(name, 200, ctypes.byref(n)))
    return n.value


def _near(got, want, a, b, factor=1.0):
    """Another order of the same sums: k terms, rounded by 2^-24 of what they add up to without signs, signs at random, six sigma."""
    a, b = (np.abs(x.data.reshape(x.shape)).astype(np.float64) for x in (a, b))
    size = a @ (b.T if b.shape[1] == a.shape[1] and b.shape[0] == want.shape[1] else b)
    off = np.abs(got.data.astype(np.float64) - want.data).reshape(want.shape)
    assert (off <= factor * 6 * 2.0 ** -24 * np.sqrt(2 * a.shape[1]) * size).all()


# slices (few rows, long contractions, the last slice shorter than the others, more to contract than columns), one piece, widths that are no
# multiple of four columns
@pytest.mark.parametrize("rows,n,k,slices", [(33, 4096, 4096, True), (40, 1024, 6000, True), (490, 768, 3072, True), (66, 2052, 4100, True), (130, 1024, 256, False), (63, 255, 3000, False),
                                             (1, 1, 1, False)])
def test_the_bits_of_the_two_calls(B, rows, n, k, slices):
    a, b, g, pre = _draw(1, rows, k), _draw(2, n, k), _draw(3, k, n), _draw(4, rows, n)
    want = B.matmulTransposed(a, b)
    assert (_slices(B) > 1) == slices
    act, mm = B.matmulTransposedGeluSaved(a, b)
    assert (_slices(B) > 1) == slices
    assert np.array_equal(mm.data, want.data) and np.array_equal(act.data, B.gelu(want).data)
    down = B.geluBackward(pre, B.matmul(a, g))
    assert np.array_equal(B.matmulGeluBackward(a, g, pre).data, down.data)


@pytest.mark.parametrize("rows,n,k", [(88, 2048, 512), (1, 4096, 1024), (490, 256, 1024)])
def test_one_piece_where_slices_gain_little(B, rows, n, k):
    """gelu and its derivative are at most 1.13 times as far off as what they are taken of."""
    a, b, g, pre = _draw(1, rows, k), _draw(2, n, k), _draw(3, k, n), _draw(4, rows, n)
    want = B.matmulTransposed(a, b)
    assert _slices(B) > 1
    act, mm = B.matmulTransposedGeluSaved(a, b)
    assert _slices(B) == 1
    _near(mm, want, a, b)
    _near(act, B.gelu(want), a, b, 1.13)
    down = B.geluBackward(pre, B.matmul(a, g))
    _near(B.matmulGeluBackward(a, g, pre), down, a, g, 1.13)


def test_infinite_and_large_values_in_slices(B):
    """Pre-activations past the cube's range, infinities and NaN: as the two calls."""
    a, b, pre = _draw(1, 64, 4096), _draw(2, 512, 4096), _draw(4, 64, 512)
    a.data[:4096] *= np.float32(1e13)
    a.data[4096] = np.inf
    a.data[2 * 4096] = np.nan
    pre.data[:5] = (1e13, -1e13, np.inf, -np.inf, np.nan)
    act, mm = B.matmulTransposedGeluSaved(a, b)
    want = B.matmulTransposed(a, b)
    assert _slices(B) > 1
    assert np.array_equal(mm.data, want.data, equal_nan=True) and np.array_equal(act.data, B.gelu(want).data, equal_nan=True)
    g = _draw(3, 4096, 512)
    got = B.matmulGeluBackward(a, g, pre)
    assert _slices(B) > 1
    assert np.array_equal(got.data, B.geluBackward(pre, B.matmul(a, g)).data, equal_nan=True)


def test_one_piece_on_the_side_stream(B):
    a, b = _draw(1, 64, 4096), _draw(2, 512, 4096)
    out, pre = B._new([64, 512]), B._new([64, 512])
    pa, pb, po, pp = (B._ptr(t) for t in (a, b, out, pre))
    call = lambda: B._gemm(ffi.GEMM_NT, pa, pb, po, 64, 512, 4096, 4096, 4096, 512, epilogue=ffi.EPI_GELU, aux=pp)
    call()
    assert _slices(B) > 1
    want = np.array(B._download(pre))
    ffi.check(B.lib.ah_side_begin())
    call()
    ffi.check(B.lib.ah_side_end())
    ffi.check(B.lib.ah_side_join())
    assert _slices(B) == 1
    _near(pre, TensorData((64, 512), "f32", want), a, b)
