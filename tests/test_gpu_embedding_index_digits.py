"""The order of positions by id where the number of digits that are sorted changes: the last id of a power of two and the first of the
next, one and no position out of range, full and partial blocks of positions."""
import numpy as np
import pytest

from alpha2_amd import _ffi as ffi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def B():
    from alpha2_amd import HipBackend
    return HipBackend(0)


@pytest.mark.parametrize("vocab", [1, 2, 15, 16, 17, 255, 256, 257, 4096, 4097, 50304, 65534])
@pytest.mark.parametrize("n", [513, 1024, 1500, 2048, 4095, 8192, 10240, 16384])
@pytest.mark.parametrize("outside", [0, 1])
def test_order(B, n, vocab, outside):
    rng = np.random.default_rng(n + vocab)
    ids = rng.integers(0, vocab, n).astype(np.int32)
    ids[rng.integers(0, n, 5)] = vocab - 1
    if outside:
        ids[rng.integers(0, n)] = vocab if n % 2 else -1
    out = B._new([B.lib.ah_embedding_index_bytes(n, vocab) // 4], "i32")
    ffi.check(B.lib.ah_embedding_index(B._ptr(B.fromArray(ids, [n], "i32")), n, vocab, out._buf.ptr))
    valid = np.nonzero((ids >= 0) & (ids < vocab))[0]
    order = valid[np.argsort(ids[valid], kind="stable")]
    want = np.full(out.size, 0xFFFFFFFF, np.uint32)
    want[:len(order)] = (ids[order].astype(np.uint32) << 16) | order.astype(np.uint32)
    assert np.array_equal(out.data.view(np.uint32), want)
