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
