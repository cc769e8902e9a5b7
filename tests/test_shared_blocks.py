"""Blocks that clones share, on the CPU: the backends' bookkeeping over a stand-in for the native library whose device memory is
host memory and whose in-place calls write recognisable values.  What is checked is who owns which bytes, not the arithmetic."""
import ctypes as C
import random
import types

import numpy as np
import pytest

from alpha2_amd import _ffi as ffi


class HostLibrary:
    """The calls the in-place operations make.  Every in-place kernel sets each element it writes to 1000 + what was there."""

    def __init__(self):
        self.blocks, self.on_alloc, self.refuse_copy = {}, None, False

    def ah_init(self, device):
        return 0

    def ah_last_error(self):
        return b"refused"

    def ah_alloc(self, nbytes, out):
        block = C.create_string_buffer(max(16, int(nbytes)) + 16)
        address = (C.addressof(block) + 15) & ~15               # (16-byte aligned, as device blocks are)
        self.blocks[address] = block
        out._obj.value = address
        if self.on_alloc is not None:
            hook, self.on_alloc = self.on_alloc, None
            hook()
        return 0

    def ah_free(self, address):
        del self.blocks[address]                                # a second free of a block is a KeyError
        return 0

    def ah_copy(self, dst, src, nbytes):
        if self.refuse_copy:
            return 4
        C.memmove(dst, src, nbytes)
        return 0

    def ah_upload(self, dst, host, nbytes):
        C.memmove(dst, host, nbytes)
        return 0

    def ah_download(self, host, src, nbytes):
        C.memmove(host, src, nbytes)
        return 0

    @staticmethod
    def view(address, n, kind=np.float32):
        return np.frombuffer((C.c_char * (n * np.dtype(kind).itemsize)).from_address(address), dtype=kind)

    def touch(self, n, *addresses):
        for p in addresses:
            self.view(p, n)[:] += 1000
        return 0

    def ah_add_inplace(self, a, b, n):
        self.view(a, n)[:] += self.view(b, n)
        return 0

    def ah_binary(self, op, a, b, out, n):
        assert op == ffi.ADD
        self.view(out, n)[:] = self.view(a, n) + self.view(b, n)
        return 0

    def ah_add_bf16(self, a, b, out, n):                        # (bf16 words added as whole numbers: not the kernel's arithmetic)
        self.view(out, n, np.uint16)[:] = self.view(a, n, np.uint16) + self.view(b, n, np.uint16)
        return 0

    def ah_scale_inplace(self, a, s, n):
        return self.touch(n, a)

    def ah_adamw(self, p, g, m, v, n, *rest):
        return self.touch(n, p, m, v)

    def ah_adamw_list(self, items, count, *rest):
        for q in items[:count]:
            self.touch(q.n, q.p, q.m, q.v)
        return 0

    def ah_lion(self, p, g, m, n, *rest):
        return self.touch(n, p, m)

    def ah_sgd(self, p, g, n, *rest):
        return self.touch(n, p)

    def ah_adafactor_2d(self, p, g, vr, vc, rows, cols, *rest):
        return self.touch(rows * cols, p) or self.touch(rows, vr) or self.touch(cols, vc)

    def ah_adafactor_flat(self, p, g, v, n, *rest):
        return self.touch(n, p, v)

    def ah_token_windows(self, corpus, n, starts, rows, cols, inputs, targets):
        first = self.view(starts, rows, np.int64)
        tokens = self.view(corpus, n, np.int32)
        at = (first[:, None] + np.arange(cols)) % n
        self.view(inputs, rows * cols, np.int32)[:] = tokens[at].reshape(-1)
        self.view(targets, rows * cols, np.int32)[:] = tokens[(at + 1) % n].reshape(-1)
        return 0

    def ah_step_kick(self):
        return 0

    def ah_sync(self):
        return 0


@pytest.fixture
def lib(monkeypatch):
    lib = HostLibrary()
    monkeypatch.setattr(ffi, "load", lambda: lib)
    return lib


def _backend(kind):
    from alpha2_amd import FastHipBackend, HipBackend
    return FastHipBackend(0) if kind == "fast" else HipBackend(0)


def _floats(B, n, seed, shape=None):
    from alpha2_amd.backend import TensorData
    t = TensorData(shape or (n,), "f32", np.random.RandomState(seed).randn(n).astype(np.float32))
    B._ptr(t)
    return t


def _device(lib, B, t):
    """What the device holds for `t`, past any copy on the host."""
    t._host_valid = False
    return np.array(t.data)


@pytest.mark.parametrize("kind", ["f32", "fast"])
@pytest.mark.parametrize("packed", [False, True])
def test_a_cloned_batch_survives_the_batches_that_follow(lib, kind, packed):
    from alpha2_amd.train import DataLoader
    B = _backend(kind)
    draws = types.SimpleNamespace(next=random.Random(3).random)
    loader = DataLoader(B, np.arange(500), draws, 2, 5, packed=packed)
    kept = []
    for _ in range(6):
        x, y = loader.nextBatch()
        cx, cy = B.clone(x), B.clone(y)
        kept.append((cx, cy, np.array(_device(lib, B, x)), np.array(_device(lib, B, y))))
        assert np.array_equal(kept[-1][3] % 500, (kept[-1][2] + 1) % 500)
        for cx, cy, wx, wy in kept:
            assert np.array_equal(_device(lib, B, cx), wx) and np.array_equal(_device(lib, B, cy), wy)
    assert len({tuple(wx) for _, _, wx, _ in kept}) == 6


def _in_place_calls(B):
    """name -> (sizes of the operands, the call, which operands it writes)."""
    one = (12,)
    return {
        "addInplace": ((one, one), lambda a, b: B.addInplace(a, b), (0,)),
        "scaleInplace": ((one,), lambda a: B.scaleInplace(a, 2.0), (0,)),
        "adamwStep": ((one,) * 4, lambda p, g, m, v: B.adamwStep(p, g, m, v, 1e-3, 0.9, 0.95, 1e-8, 0.0, 0.1, 0.05), (0, 2, 3)),
        "lionStep": ((one,) * 3, lambda p, g, m: B.lionStep(p, g, m, 1e-3, 0.9, 0.99, 0.0), (0, 2)),
        "sgdStep": ((one,) * 2, lambda p, g: B.sgdStep(p, g, 0.1), (0,)),
        "adafactorStep2d": (((3, 4), (3, 4), (3,), (4,)), lambda p, g, r, c: B.adafactorStep2d(p, g, r, c, 1e-3, 0.9, 1e-8, 1.0, 0.0), (0, 2, 3)),
        "adafactorStepFlat": ((one,) * 3, lambda p, g, v: B.adafactorStepFlat(p, g, v, 1e-3, 0.9, 1e-8, 1.0, 0.0), (0, 2)),
    }


@pytest.mark.parametrize("writer", ["f32", "fast"])
@pytest.mark.parametrize("name", ["addInplace", "scaleInplace", "adamwStep", "lionStep", "sgdStep", "adafactorStep2d", "adafactorStepFlat"])
@pytest.mark.parametrize("side", ["original", "clone"])
def test_in_place_calls_leave_the_other_side_of_a_clone_alone(lib, writer, name, side):
    """Clones made by the fp32 backend, written through either backend, from either side."""
    maker, B = _backend("f32"), _backend(writer)
    shapes, call, written = _in_place_calls(B)[name]
    originals = [_floats(maker, int(np.prod(s)), i, s) for i, s in enumerate(shapes)]
    before = [np.array(t.data) for t in originals]
    clones = [maker.clone(t) for t in originals]
    operands, others = (originals, clones) if side == "original" else (clones, originals)
    call(*operands)
    B.syncGpu()
    for i, (t, o) in enumerate(zip(operands, others)):
        assert np.array_equal(_device(lib, maker, o), before[i]), i
        assert np.array_equal(_device(lib, maker, t), before[i]) == (i not in written), i


@pytest.mark.parametrize("side", ["original", "clone"])
def test_bf16_add_in_place_leaves_the_other_side_of_a_clone_alone(lib, side):
    maker, B = _backend("f32"), _backend("fast")
    a, b = B._new((16,), "f32", "bf16"), B._new((16,), "f32", "bf16")
    lib.view(a._buf.ptr, 16, np.uint16)[:] = np.arange(16) + 16256
    lib.view(b._buf.ptr, 16, np.uint16)[:] = 1
    c = maker.clone(a)
    w, other = (a, c) if side == "original" else (c, a)
    B.addInplace(w, b)
    assert np.array_equal(lib.view(other._buf.ptr, 16, np.uint16), np.arange(16) + 16256)
    assert np.array_equal(lib.view(w._buf.ptr, 16, np.uint16), np.arange(16) + 16257)


@pytest.mark.parametrize("moment", ["while the writer's block is made", "before"])
def test_the_shared_block_is_freed_by_whoever_leaves_it_last(lib, moment):
    """The other side may be collected inside the writer's own allocation: the block has no owner then once the writer has moved."""
    B = _backend("f32")
    a = _floats(B, 12, 1)
    want = np.array(a.data)
    held = [B.clone(a)]
    if moment == "before":
        held.clear()
    else:
        lib.on_alloc = held.clear
    B.scaleInplace(a, 2.0)
    assert np.array_equal(_device(lib, B, a), want + 1000) and len(lib.blocks) == 1
    B.releaseGpuTensor(a)
    assert not lib.blocks


def test_a_refused_copy_leaves_both_sides_as_they_were(lib):
    B = _backend("f32")
    a = _floats(B, 12, 1)
    want, c = np.array(a.data), B.clone(a)
    lib.refuse_copy = True
    with pytest.raises(Exception):
        B.scaleInplace(a, 2.0)
    assert len(lib.blocks) == 1 and a._buf.ptr == c._buf.ptr
    lib.refuse_copy = False
    B.scaleInplace(a, 2.0)
    assert np.array_equal(_device(lib, B, a), want + 1000) and np.array_equal(_device(lib, B, c), want)
