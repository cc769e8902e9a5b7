"""residual + A B^T from one call: against the two calls it stands for (same sums in the same order, so the same bits), with its gradients,
the MLP that ends in one, and in one piece on the side stream."""
import ctypes

import numpy as np
import pytest

from alpha2_amd import _ffi as ffi
from alpha2_amd import autograd as ag
from alpha2_amd.autograd import Ctx, Tape, Variable

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def B():
    from alpha2_amd import HipBackend
    return HipBackend(0)


def _inputs(B, rows, n, k, lead=()):
    rng = np.random.default_rng(rows + n + k)
    draw = lambda *s: B.fromArray(rng.standard_normal(s).astype(np.float32).ravel().tolist(), list(s))
    return draw(rows, k), draw(n, k), draw(*lead, rows // (int(np.prod(lead)) if lead else 1), n)


def _check(got, a, b, r):
    """Against 64 bits.  Bound: k products and additions rounded by 2^-24 of at most sum |a| |b| each, signs at random, six sigma
    (the bit-for-bit comparison is the sharp one; a lost slice or residual is off by far more)."""
    a, b, r = (np.asarray(t.data, np.float64).reshape(-1, t.shape[-1]) for t in (a, b, r))
    size = np.abs(a) @ np.abs(b).T
    error = np.abs(np.asarray(got.data, np.float64).reshape(r.shape) - (a @ b.T + r))
    assert (error <= 6 * 2.0 ** -24 * (np.sqrt(a.shape[1] + 1) * size + np.abs(r))).all()


# one piece and slices (few tiles, a long contraction), odd widths and rows, a single row and element
@pytest.mark.parametrize("rows,n,k", [(1, 1, 1), (1, 256, 1024), (17, 255, 33), (63, 64, 3072), (128, 128, 512), (490, 768, 3072), (2048, 256, 64), (130, 132, 17)])
def test_same_bits_as_the_two_calls(B, rows, n, k):
    a, b, r = _inputs(B, rows, n, k)
    got = B.matmulTransposedAdd(a, b, r)
    want = B.add(r, B.matmulTransposed(a, b))
    assert got.shape == want.shape and np.array_equal(np.asarray(got.data), np.asarray(want.data))
    _check(got, a, b, r)


def test_other_shapes_are_left_to_the_two_calls(B):
    a, b, r = _inputs(B, 6, 8, 4)
    assert B.matmulTransposedAdd(a, b, B.reshape(r, [8, 6])) is None
    assert B.matmulTransposedAdd(B.reshape(a, [2, 3, 4]), b, r) is None
    assert B.matmulTransposedAdd(B.reshape(a, [4, 6]), b, r) is None


def test_gradients(B):
    def run(product):
        a, b, r = (Variable(t, True) for t in _inputs(B, 34, 48, 72, lead=(2,)))
        ctx = Ctx(Tape(), B)
        y = product(ctx, r, a, b)
        loss = ag.sum(ctx, ag.mul(ctx, y, y))
        ctx.tape.backward(loss, B, B.releaseGpuTensor)
        return [np.array(v.grad.data) for v in (a, b, r)]
    one = run(lambda c, r, a, b: ag.residualProduct(c, r, a, b, 0.3, False))
    two = run(lambda c, r, a, b: ag.add(c, r, ag.reshape(c, ag.matmulTransposed(c, a, b), r.data.shape)))
    for g, w in zip(one, two):
        assert np.array_equal(g, w)


def test_one_piece_on_the_side_stream(B):
    a, b, r = _inputs(B, 64, 64, 3072)
    out = B._new([64, 64])
    pa, pb, pr, po = (B._ptr(t) for t in (a, b, r, out))
    call = lambda: B._gemm(ffi.GEMM_NT, pa, pb, po, 64, 64, 3072, 3072, 3072, 64, epilogue=ffi.EPI_RESIDUAL, aux=pr)
    slices = ctypes.c_int32()
    name = ctypes.create_string_buffer(200)

    def pieces():
        ffi.check(B.lib.ah_gemm_last_kernel(name, 200, ctypes.byref(slices)))
        return slices.value
    call()
    assert pieces() > 1
    ffi.check(B.lib.ah_side_begin())
    call()
    ffi.check(B.lib.ah_side_end())
    ffi.check(B.lib.ah_side_join())
    assert pieces() == 1
    _check(out, a, b, r)


@pytest.mark.parametrize("rows,width,hidden", [(34, 48, 192), (2, 4, 4), (130, 256, 1024), (66, 96, 40)])      # the last: no wider than the input
@pytest.mark.parametrize("scale", [1.0, 1e13])                     # 1e13: pre-activations whose cube is past f32
def test_gelu_mlp_has_the_bits_of_its_parts(B, rows, width, hidden, scale):
    def run(op):
        rng = np.random.default_rng(rows)
        draw = lambda k, *s: Variable(B.fromArray((k * rng.standard_normal(s)).astype(np.float32).ravel(), list(s)), True)
        v = draw(1.0, 2, rows // 2, width), draw(scale, rows, width), draw(1.0, hidden, width), draw(1.0, width, hidden)
        ctx = Ctx(Tape(), B)
        y = op(ctx, *v)
        ctx.tape.backward(ag.sum(ctx, ag.scale(ctx, y, 0.5)), B, B.releaseGpuTensor)
        return [np.array(t.grad.data) for t in v]
    one = run(lambda c, r, x, a, b: ag.geluMlp(c, r, x, a, b, 0.0, True))
    two = run(lambda c, r, x, a, b: ag.add(c, r, ag.reshape(c, ag.matmulTransposed(c, ag.gelu(c, ag.matmulTransposed(c, x, a)), b), r.data.shape)))
    for g, w in zip(one, two):
        assert np.isfinite(w).all() and np.array_equal(g, w)
