"""Groups of weight gradients on tiles of 128, 192 and 256 columns: ragged edges, halves of k, accumulation and the sum of squares."""
import ctypes as C

import numpy as np
import pytest

from alpha2_amd import _ffi as ffi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def B():
    from alpha2_amd import HipBackend
    return HipBackend(0)


@pytest.mark.parametrize("shapes,K,width", [
    ([(264, 136), (8, 8), (256, 128), (248, 120)], 128, 2),          # every problem in two halves
    ([(264, 136), (520, 384)], 192, 2),                              # whole (k is not halves of 64)
    ([(2552, 376)] + 4 * [(2560, 384)], 128, 3),
    ([(2552, 392)] + 8 * [(2560, 384)], 64, 3),
    ([(4096, 4088)], 64, 4),
])
def test_widths(B, shapes, K, width):
    """The operands are whole numbers up to 8, so every product and sum is exact in fp32 (at most 192 x 64 twice, and the square of no sum passes 2^53
    in 64 bits); the sum of squares is added up in fp32 inside a wave: 2^-24 for each of at most 2^7 additions after one another."""
    rs = np.random.RandomState(K + len(shapes))
    keep, descs, outs, wants = [], [], [], []
    for m, n in shapes:
        a, b = rs.randint(-8, 9, (K, m)).astype(np.float32), rs.randint(-8, 9, (K, n)).astype(np.float32)
        ta, tb = (B.castStore(B.fromArray(t.reshape(-1), list(t.shape)), "bf16") for t in (a, b))
        out = B.full((m, n), 5.0)
        keep += [ta, tb]
        outs.append(out)
        wants.append(a.astype(np.float64).T @ b.astype(np.float64))
        descs.append(ffi.AhGemm(ffi.GEMM_TN, ffi.BF16, ffi.F32, ffi.EPI_NONE, m, n, K, m, n, n, 1, 0, 0, 0, B._ptr(ta), B._ptr(tb), B._ptr(out), 0))
    arr, plan = (ffi.AhGemm * len(descs))(*descs), C.c_uint64()
    ffi.check(B.lib.ah_gemm_grouped_plan(arr, len(descs), C.byref(plan)))
    for epilogue, times in ((ffi.EPI_NONE, 1), (ffi.EPI_ACCUM, 2), (ffi.EPI_ACCUM, 3)):
        total = B.full((1,), 0.0)
        if times == 3:
            ffi.check(B.lib.ah_gemm_grouped_update(plan.value, arr, len(descs)))
            ffi.check(B.lib.ah_gemm_grouped_run(plan.value, epilogue))
        else:
            ffi.check(B.lib.ah_gemm_grouped_run_sumsq(plan.value, epilogue, B._ptr(total)))
        assert ", %d, " % width in B.lastGemmKernel()[0]
        for out, want in zip(outs, wants):
            B._dirty(out)
            assert np.array_equal(out.data.reshape(want.shape), times * want)
        if times < 3:
            B._dirty(total)
            want = sum(float(((times * w) ** 2).sum()) for w in wants)
            assert abs(float(total.data[0]) - want) <= 2.0 ** -17 * want
    ffi.check(B.lib.ah_gemm_grouped_destroy(plan.value))


@pytest.mark.parametrize("shapes,narrow", [
    ([(4096, 384)] + 8 * [(1152, 384), (384, 384), (1536, 384), (384, 1536)], False),      # 336 tiles at 256 columns: the last 80 and more in halves
    ([(1000, 320)] + 6 * [(960, 320), (320, 320), (1280, 320), (320, 1280)], True),
    (6 * [(520, 384), (264, 136)], True),
    ([(2552, 376)] + 8 * [(2560, 384)], True),                                              # 180 tiles: none
])
def test_a_tiles_width_halves_no_other_problem(B, shapes, narrow):
    """Which products are added up in two halves of k follows from the tiles at 256 columns, whatever width is taken.  Each result is 2^24 in the first half
    of k and two ones in the second, a step of the matrix instruction apart: 2^24 + 2 from halves, and 2^24 where each one is lost beside it."""
    tiles = [-(-m // 256) * -(-n // 256) for m, n in shapes]
    tail, halved, total = sum(tiles) % 256, set(), 0
    if 0 < tail <= 128:
        for i in reversed(range(len(shapes))):
            if total < tail and total + tiles[i] <= 128:
                halved.add(i)
                total += tiles[i]
    assert total >= tail or tail > 128
    K, at, descs, outs, keep = 128, [0, 64, 112], [], [], []
    for m, n in shapes:
        a, b = np.zeros((K, m), np.float32), np.zeros((K, n), np.float32)
        for t in (a, b):
            t[at] = np.array([[4096.0], [1.0], [1.0]])
        ta, tb = (B.castStore(B.fromArray(t.reshape(-1), list(t.shape)), "bf16") for t in (a, b))
        outs.append(B._new((m, n)))
        keep += [ta, tb]
        descs.append(ffi.AhGemm(ffi.GEMM_TN, ffi.BF16, ffi.F32, ffi.EPI_NONE, m, n, K, m, n, n, 1, 0, 0, 0, B._ptr(ta), B._ptr(tb), B._ptr(outs[-1]), 0))
    arr, plan = (ffi.AhGemm * len(descs))(*descs), C.c_uint64()
    ffi.check(B.lib.ah_gemm_grouped_plan(arr, len(descs), C.byref(plan)))
    ffi.check(B.lib.ah_gemm_grouped_run(plan.value, ffi.EPI_NONE))
    assert (", 4, " not in B.lastGemmKernel()[0]) == narrow
    for i, out in enumerate(outs):
        B._dirty(out)
        assert np.all(out.data == 2.0 ** 24 + (2 if i in halved else 0)), i
    ffi.check(B.lib.ah_gemm_grouped_destroy(plan.value))
