"""residualDropoutAdd with the LayerNorm behind it, and a LayerNorm's backward pass with the mask multiply behind it, against the passes one by one: the
same bits."""
import numpy as np
import pytest

from alpha2_amd import _ffi as ffi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def B():
    from alpha2_amd import HipBackend
    return HipBackend(0)


# a row's quads on both sides of a wave's multiples, one seed and several (the last with fewer rows), elements past 4.0 M, where the mask's hash leaves whole numbers
@pytest.mark.parametrize("rows,per_seed,dim", [(1, 1, 4), (5, 5, 252), (7, 3, 256), (33, 33, 260), (2050, 1025, 384), (130, 64, 768), (64, 64, 1024), (31, 8, 1028),
                                               (9, 9, 1540), (2200, 2200, 2048)])
@pytest.mark.parametrize("residual_grad", [True, False])
def test_one_pass_has_the_bits_of_two(B, rows, per_seed, dim, residual_grad):
    rs, n, lib, check = np.random.RandomState(rows + dim), rows * dim, B.lib, ffi.check
    seeds = B.fromArray(rs.randint(-1000, 1 << 30, -(-rows // per_seed)).astype(np.int32), [-(-rows // per_seed)], "i32")
    bf = lambda: B.castStore(B.fromArray(rs.randn(n).astype(np.float32), [n]), "bf16")
    x, res, g = bf(), bf(), bf()
    w, b = (B.fromArray((1 + 0.3 * rs.randn(dim)).astype(np.float32), [dim]) for _ in range(2))
    new = lambda: B._new((n,), "f32", "bf16")
    p, parts = B._ptr, int(lib.ah_layernorm_bwd_partials_bytes(rows, dim)) // 4
    counter, prob = 5, 0.3

    def masked(src, add, dst):
        for s in range(seeds.size):
            at, m = s * per_seed * dim * 2, min(per_seed, rows - s * per_seed) * dim
            check(lib.ah_dropout_apply(p(src) + at, ffi.BF16, p(add) + at if add is not None else 0, p(dst) + at, ffi.BF16, m, p(seeds) + 4 * s, counter, prob))

    stream, out, stream2, out2 = new(), new(), new(), new()
    masked(x, res, stream)
    check(lib.ah_layernorm(p(stream), p(w), p(b), p(out), rows, dim, 1e-5, ffi.BF16, ffi.BF16))
    check(lib.ah_dropout_layernorm(p(x), p(res), p(stream2), p(w), p(b), p(out2), rows, dim, 1e-5, p(seeds), per_seed, counter, prob))
    dx, drop, dx2, drop2, sums, sums2 = new(), new(), new(), new(), B._new((parts,)), B._new((parts,))
    dxf, dxf2 = B._new((n,)), B._new((n,))
    add = p(res) if residual_grad else 0
    check(lib.ah_layernorm_bwd_deferred(p(stream), p(w), p(g), ffi.BF16, add, p(dxf), p(dx), p(sums), rows, dim, 1e-5, ffi.BF16))
    masked(dx, None, drop)
    check(lib.ah_layernorm_bwd_dropout(p(stream), p(w), p(g), add, p(dxf2), p(dx2), p(drop2), p(sums2), rows, dim, 1e-5, p(seeds), per_seed, counter, prob))
    for a, c, what in ((stream, stream2, "stream"), (out, out2, "out"), (dx, dx2, "dx"), (drop, drop2, "dropped"), (sums, sums2, "sums"), (dxf, dxf2, "dx in f32")):
        B._dirty(a), B._dirty(c)
        a, c = np.array(a.data), np.array(c.data)
        assert np.array_equal(a.view(np.uint32), c.view(np.uint32)), what


def test_refusals(B):
    lib, a = B.lib, 1 << 20
    call = lambda rows=4, dim=8, per=4, p=0.1, x=a, seeds=a: lib.ah_dropout_layernorm(x, a, a, a, a, a, rows, dim, 1e-5, seeds, per, 0, p)
    back = lambda rows=4, dim=8, per=4, p=0.1, x=a, seeds=a: lib.ah_layernorm_bwd_dropout(x, a, a, 0, 0, a, a, a, rows, dim, 1e-5, seeds, per, 0, p)
    for f in (call, back):
        for bad in (dict(rows=0), dict(dim=6), dict(dim=2052), dict(per=0), dict(per=1 << 30), dict(p=1.0), dict(x=0), dict(x=a + 4), dict(seeds=0), dict(seeds=a + 2)):
            assert f(**bad) == 2, bad
