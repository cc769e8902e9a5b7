"""fp32 attention where its scores lie on both sides of the line between the two forms of tanh (0.625 of the cap) and in tiles with and
without masked scores, against the same function in 64 bits."""
import ctypes as C
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def B():
    from alpha2_amd import HipBackend
    return HipBackend(0)


def _exact(q, k, v, g, scale, cap):
    """O, dQ, dK, dV, and the norms of what is summed for each, without its signs."""
    s = q @ k.transpose(0, 2, 1) * scale
    t = np.tanh(s / cap) if cap > 0 else 0 * s
    s = cap * t if cap > 0 else s
    T = q.shape[1]
    s = np.where(np.tril(np.ones((T, T), bool)), s, -np.inf)
    p = np.exp(s - s.max(2, keepdims=True))
    p /= p.sum(2, keepdims=True)
    o, vt = p @ v, v.transpose(0, 2, 1)
    ds = p * (g @ vt - (g * o).sum(2, keepdims=True)) * (1 - t * t)
    terms = p * (abs(g) @ abs(vt) + abs(g * o).sum(2, keepdims=True)) * (1 - t * t)
    sizes = [np.linalg.norm(x) for x in (p @ abs(v), terms @ abs(k) * scale, terms.transpose(0, 2, 1) @ abs(q) * scale, p.transpose(0, 2, 1) @ abs(g))]
    return (o, ds @ k * scale, ds.transpose(0, 2, 1) @ q * scale, p.transpose(0, 2, 1) @ g), sizes, float(np.abs(np.where(np.isfinite(s), s, 0)).max())


@pytest.mark.parametrize("heads,T,D", [(3, 1, 8), (3, 31, 32), (2, 33, 64), (2, 129, 24), (40, 160, 48), (2, 300, 32), (300, 130, 64)])
@pytest.mark.parametrize("cap", [0.0, 0.75, 30.0])
@pytest.mark.parametrize("spread", [0.3, 3.0, 25.0])
def test_scores_on_both_sides_of_the_cap(B, heads, T, D, cap, spread):
    """Bound, against the sums without signs: some ten roundings in a row on the way to a result, and two of a score's (its product's
    and tanh's), which its size multiplies in the exponential, 2^-24 each."""
    from alpha2_amd import _ffi as ffi
    from alpha2_amd.backend import TensorData
    rs = np.random.default_rng(T + D)
    a = [rs.standard_normal((heads, T, D), dtype=np.float32) for _ in range(4)]
    a[0] *= np.float32(spread)
    t = [TensorData(x.shape, "f32", x) for x in a]
    out = [B._new(a[0].shape) for _ in range(4)]
    lse = B._new((heads, T))
    st = (heads * T * D, T * D, D)
    scale = 1 / math.sqrt(D)
    p = [B._ptr(x) for x in t]
    f = ffi.AhFlash(ffi.F32, 1, heads, T, D, *st, *st, *st, *st, scale, cap, p[0], p[1], p[2], out[0]._buf.ptr, lse._buf.ptr, p[3],
                    out[1]._buf.ptr, out[2]._buf.ptr, out[3]._buf.ptr, 0, 0)
    ffi.check(B.lib.ah_flash_fwd(C.byref(f)))
    ffi.check(B.lib.ah_flash_bwd(C.byref(f)))
    want, sizes, largest = _exact(*(x[:4].astype(np.float64) for x in a), scale, cap)
    for name, got, w, size in zip(("O", "dQ", "dK", "dV"), out, want, sizes):
        off = np.linalg.norm(got.data.reshape(a[0].shape)[:4].astype(np.float64) - w)
        assert off <= (10 + 2 * largest) * 2.0 ** -24 * size, (name, off / size * 2 ** 24)


@pytest.mark.parametrize("cap", [1e-39, 2.0 ** -149, 1e-37])
@pytest.mark.parametrize("heads,T,D", [(2, 40, 32), (300, 130, 64), (2, 33, 128)])
def test_scores_of_zero_under_the_smallest_caps(B, heads, T, D, cap):
    """Down to caps whose inverse is past the range: a score of zero stays one, others weigh the same to 2^-24.  Row 3 of the queries is zero,
    which a derivative passes (tanh' 0 = 1); at the others, scores of a unit or so, it is nothing.  Bound as above."""
    from alpha2_amd import _ffi as ffi
    from alpha2_amd.backend import TensorData
    rs = np.random.default_rng(T + D)
    a = [rs.standard_normal((heads, T, D), dtype=np.float32) for _ in range(4)]
    a[0][:, 3] = 0
    t = [TensorData(x.shape, "f32", x) for x in a]
    out = [B._new(a[0].shape) for _ in range(4)]
    lse = B._new((heads, T))
    st = (heads * T * D, T * D, D)
    p = [B._ptr(x) for x in t]
    f = ffi.AhFlash(ffi.F32, 1, heads, T, D, *st, *st, *st, *st, 1.0, cap, p[0], p[1], p[2], out[0]._buf.ptr, lse._buf.ptr, p[3],
                    out[1]._buf.ptr, out[2]._buf.ptr, out[3]._buf.ptr, 0, 0)
    ffi.check(B.lib.ah_flash_fwd(C.byref(f)))
    ffi.check(B.lib.ah_flash_bwd(C.byref(f)))
    want, sizes, _ = _exact(*(x[:4].astype(np.float64) for x in a), 1.0, float(np.float32(cap)))
    for name, got, w, size in zip(("O", "dQ", "dK", "dV"), out, want, sizes):
        off = np.linalg.norm(got.data.reshape(a[0].shape)[:4].astype(np.float64) - w)
        assert off <= 10 * 2.0 ** -24 * size, (name, off / size * 2 ** 24)
