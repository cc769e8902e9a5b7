"""Cross-entropy where the number of threads to a row changes, and the embedding's gradient where an id's positions fill many blocks of 32."""
import numpy as np
import pytest

from alpha2_amd import _ffi as ffi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def B():
    from alpha2_amd import HipBackend
    return HipBackend(0)


@pytest.mark.parametrize("dtype,c", [("f32", c) for c in (1, 3, 4, 127, 129, 255, 256, 1023, 1024, 1025, 1028, 2048)] +
                         [("bf16", c) for c in (1, 8, 127, 129, 504, 512, 520, 1023, 1024, 1032, 2040, 2047, 2048, 2049, 2056, 8184, 8192, 8200, 16384, 16392)])
@pytest.mark.parametrize("n", [1, 3, 4, 70])
def test_rows_of_every_number_of_threads(B, dtype, c, n):
    """Against 64 bits on the logits as stored.  A thread adds up to 40 terms after one another, thirteen more join them with three roundings each, and
    each exponential is within 2^-21 of its own (an argument of up to 24 in 2^-24 steps, and the instruction's last place): the sum is within 2^-17.5,
    the log of it that much beside the roundings of values up to 24.  A probability adds the rounding of its argument; the one taken from
    it, the scale (two roundings) and the product are four of the result."""
    code, rs = ffi.DTYPE_CODE[dtype], np.random.RandomState(c + n)
    lg = (rs.randn(n, c) * 3).astype(np.float32)
    tg = rs.randint(0, c, n).astype(np.int32)
    tg[0] = c - 1
    src, tgd = B.castStore(B.fromArray(lg.reshape(-1), [n, c]), dtype), B.fromArray(tg, [n], "i32")
    x = np.array(src.data, dtype=np.float64).reshape(n, c)
    top = x.max(1, keepdims=True)
    lse = top + np.log(np.exp(x - top).sum(1, keepdims=True))
    want = np.exp(x - lse)
    want[np.arange(n), tg] -= 1
    want *= 0.7 / n
    loss, ld, dl, dl1 = B._new(()), B._new((n,)), B._new((n, c), "f32", dtype), B._new((n, c), "f32", dtype)
    ffi.check(B.lib.ah_cross_entropy(B._ptr(src), code, B._ptr(tgd), B._ptr(loss), B._ptr(ld), n, c))
    ffi.check(B.lib.ah_cross_entropy_bwd(B._ptr(src), code, B._ptr(tgd), B._ptr(ld), 0, 0.7, B._ptr(dl), n, c))
    ffi.check(B.lib.ah_cross_entropy_fwd_bwd(B._ptr(src), code, B._ptr(tgd), B._ptr(loss), B._ptr(ld), 0, 0.7, B._ptr(dl1), n, c))
    for t in (loss, ld, dl, dl1):
        B._dirty(t)
    eps = 2.0 ** -17
    assert np.all(np.abs(np.array(ld.data, np.float64) - lse[:, 0]) <= eps)
    assert abs(float(loss.data[0]) - float((lse[:, 0] - x[np.arange(n), tg]).mean())) <= 2 * eps
    got = np.array(dl.data, np.float64).reshape(n, c)
    half = 2.0 ** -22 + (2.0 ** -8 if dtype == "bf16" else 0.0)
    assert np.all(np.abs(got - want) <= np.abs(want) * half + (np.exp(x - lse) + 2.0 ** -24) * (0.7 / n) * 2 * eps)
    assert np.array_equal(np.array(dl1.data), np.array(dl.data))


@pytest.mark.parametrize("dtype,c,more", [("f32", c, 4096) for c in (252, 256, 260, 512, 516, 1000, 1024, 1028)] +
                         [("bf16", c, 20000) for c in (504, 512, 520, 1024, 1032, 2040, 2048, 2056, 4096, 4104, 8192, 8200)])
def test_classes_of_no_weight_change_no_bit(B, dtype, c, more):
    """Classes whose exponential is zero, behind the others: a row's sum keeps its bits, so the number of threads that a row of c classes gets is none of
    its order of summation.  (Their terms are exact zeros, and merging with a thread that has nothing else multiplies by one and adds zero.)"""
    n, rs = 70, np.random.RandomState(c)
    lg = np.full((n, more), -3e38, np.float32)
    lg[:, :c] = rs.randn(n, c) * 3
    tg, code, got = rs.randint(0, c, n).astype(np.int32), ffi.DTYPE_CODE[dtype], []
    tgd = B.fromArray(tg, [n], "i32")
    for classes in (c, more):
        src = B.castStore(B.fromArray(np.ascontiguousarray(lg[:, :classes]).reshape(-1), [n, classes]), dtype)
        loss, ld, ld1, dl = B._new(()), B._new((n,)), B._new((n,)), B._new((n, classes), "f32", dtype)
        ffi.check(B.lib.ah_cross_entropy(B._ptr(src), code, B._ptr(tgd), B._ptr(loss), B._ptr(ld), n, classes))
        ffi.check(B.lib.ah_cross_entropy_fwd_bwd(B._ptr(src), code, B._ptr(tgd), B._ptr(loss), B._ptr(ld1), 0, 0.7, B._ptr(dl), n, classes))
        for t in (ld, ld1, dl):
            B._dirty(t)
        got.append((np.array(ld.data), np.array(ld1.data), np.array(dl.data).reshape(n, classes)[:, :c]))
    for a, b in zip(*got):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("c", [255, 256, 3000, 9001])
def test_an_infinite_logit_is_not_a_number_in_the_loss(B, dtype, c):
    """inf - inf, as in the loops the kernels stand for, in whole chunks of 16 bytes and in rows that are none."""
    lg = np.zeros((4, c), np.float32)
    lg[2, c // 2] = np.inf
    src, tgd = B.castStore(B.fromArray(lg.reshape(-1), [4, c]), dtype), B.fromArray(np.zeros(4), [4], "i32")
    loss, ld = B._new(()), B._new((4,))
    ffi.check(B.lib.ah_cross_entropy(B._ptr(src), ffi.DTYPE_CODE[dtype], B._ptr(tgd), B._ptr(loss), B._ptr(ld), 4, c))
    for t in (loss, ld):
        B._dirty(t)
    assert np.array_equal(np.isnan(ld.data), [False, False, True, False]) and np.isnan(loss.data[0])


@pytest.mark.parametrize("dim", [4, 64, 80, 256, 260, 320])
@pytest.mark.parametrize("count", [33, 64, 63 * 32, 64 * 32, 65 * 32 + 1, 130 * 32])
@pytest.mark.parametrize("before", [0, 5, 31])
def test_an_id_over_many_blocks_is_summed_in_order(B, dim, count, before):
    """Position by position inside a block of 32 of the sorted positions, then block by block."""
    n, rs = count + before + 40, np.random.RandomState(count + before)
    ids = np.concatenate([np.zeros(before), np.full(count, 1), np.full(n - count - before, 2)]).astype(np.int32)
    rs.shuffle(ids)
    g = rs.randn(n, dim).astype(np.float32)
    gw = B.embeddingBackward(B.fromArray(ids, [n], "i32"), B.fromArray(g.reshape(-1), [n, dim]), 3).data.reshape(3, dim)
    order, at = np.argsort(ids, kind="stable"), 0
    for i in range(3):
        end, total = at + int((ids == i).sum()), None
        while at < end:
            stop = min(end, (at // 32 + 1) * 32)
            part = np.zeros(dim, np.float32)
            for p in order[at:stop]:
                part = part + g[p]
            total = part if total is None else total + part
            at = stop
        assert total is None or np.array_equal(gw[i], total), i
