"""Which contexts and parameters KeptContext takes, on the CPU: over a stand-in for the native library that knows its blocks and whose
copies and rows must stay inside them."""
import ctypes as C
import types

import numpy as np
import pytest

from alpha2_amd import _ffi as ffi, decode
from alpha2_amd.autograd import Variable
from alpha2_amd.model import ModelConfig, initGPT


class HostLibrary:
    def __init__(self):
        self.blocks, self.tokens = {}, []

    def ah_init(self, device):
        return 0

    def ah_last_error(self):
        return b"refused"

    def ah_alloc(self, nbytes, out):
        block = C.create_string_buffer(int(nbytes) + 16)
        address = (C.addressof(block) + 15) & ~15
        self.blocks[address] = (int(nbytes), block)
        out._obj.value = address
        return 0

    def ah_free(self, address):
        del self.blocks[address]
        return 0

    def inside(self, address, nbytes):
        return any(a <= address and address + nbytes <= a + n for a, (n, _) in self.blocks.items())

    def ah_upload(self, dst, host, nbytes):
        assert self.inside(dst, nbytes)
        C.memmove(dst, host, nbytes)
        return 0

    def ah_download(self, host, src, nbytes):
        C.memmove(host, src, nbytes)
        return 0

    def ah_fill_f32(self, dst, value, n):
        assert self.inside(dst, 4 * n)
        return 0

    def ah_copy(self, dst, src, nbytes):
        assert self.inside(dst, nbytes) and self.inside(src, nbytes)
        return 0

    def ah_decode_head(self, model, row):
        m = model._obj
        assert self.inside(row, 4 * m.width) and self.inside(m.head, 4 * m.width * m.vocab)
        return 0

    def ah_decode(self, model, layers, token, pos):
        m = model._obj
        if not 0 <= pos < m.rows:
            return 2
        assert self.inside(m.wpe + 4 * m.width * pos, 4 * m.width) and self.inside(m.head, 4 * m.width * m.vocab)
        self.tokens.append((token, pos, m.head))
        return 0


def _model(monkeypatch, ctx, wpe_rows=None):
    from alpha2_amd import HipBackend
    monkeypatch.setattr(ffi, "load", lambda: HostLibrary())
    B = HipBackend(0)
    cfg = ModelConfig(vocabSize=20, blockSize=wpe_rows or ctx, nLayer=2, nEmbd=16, nHead=2)
    params = initGPT(cfg, B, types.SimpleNamespace(fillGauss=lambda n, std: np.full(n, std, np.float32)))
    cfg.blockSize = ctx

    def blocks(c, cfg, params, ids):
        n = ids.shape[1]
        c.keptQkv += [Variable(B._new((n, 3 * cfg.nEmbd))) for _ in params["layers"]]
        return Variable(B._new((1, n, cfg.nEmbd)))
    monkeypatch.setattr(decode, "gptBlocks", blocks)
    return B, cfg, params


# blockSize, rows of wpe, longest, the longest context that is taken: the cache has 64 rows or more, and fewer may have been asked for;
# a longest past blockSize; fewer positions than the cache has rows
@pytest.mark.parametrize("ctx,wpe,longest,most", [(64, 64, 64, 64), (200, 200, 70, 70), (40, 200, 70, 40), (128, 70, 70, 70), (200, 200, 5, 5)])
def test_a_context_past_what_was_asked_for_is_refused(monkeypatch, ctx, wpe, longest, most):
    B, cfg, params = _model(monkeypatch, ctx, wpe)
    kept = decode.KeptContext.of(cfg, params, B, longest)
    tokens = np.arange(300, dtype=np.int32) % 20
    for n in (0, most + 1, most + 7, 200):
        with pytest.raises(ValueError):
            kept.lastRow(tokens[:n], None)
    assert kept.lastRow(tokens[:most], None).shape == (20,)             # all at once
    kept.known = 0
    kept.lastRow(tokens[:most - 1], None)
    kept.lastRow(tokens[:most], None)                                   # its last token by itself
    assert B.lib.tokens[-1][1] == most - 1
    with pytest.raises(ValueError):
        kept.lastRow(tokens[:most + 1], None)
    assert kept.known == most
    kept.close()


def _sample(monkeypatch, replace, when):
    """16 tokens behind a prompt of 5 while the caller's own code replaces the head's tensor, on the way out of the pass over the prompt or in
    flushGpu; returns what the device saw of the single tokens and the contexts that were run whole."""
    from alpha2_amd import sample
    from alpha2_amd.backend import TensorData
    B, cfg, params = _model(monkeypatch, 64)
    done, whole = [], []

    def move(now):
        if now == when and not done:
            done.append(1)
            old = params["lmHead"].data
            params["lmHead"].data = replace(TensorData, old)
            B.releaseGpuTensor(old)
    release = lambda t: (B.releaseGpuTensor(t), move("release"))
    monkeypatch.setattr(sample, "_lastRow", lambda c, p, b, context, r: whole.append(context.size) or np.ones(20, np.float32))
    monkeypatch.setattr(B, "_download", lambda t: np.ones(20, np.float32))
    sample.sampleTokens(cfg, params, B, None, np.arange(5), sample.SampleConfig(steps=16, temperature=0), release, lambda: move("flush"))
    assert done
    return B, params, B.lib.tokens, whole


@pytest.mark.parametrize("when", ["release", "flush"])
def test_a_parameter_that_moves_is_followed(monkeypatch, when):
    B, params, tokens, whole = _sample(monkeypatch, lambda T, old: T(old.shape, "f32", old.data), when)
    assert [pos for _, pos, _ in tokens] == list(range(5, 20)) and not whole
    assert tokens[-1][2] == B._ptr(params["lmHead"].data)


@pytest.mark.parametrize("when", ["release", "flush"])
def test_a_parameter_of_another_shape_ends_the_kept_context(monkeypatch, when):
    """The pass over the whole context then says what it thinks of it, as it does for every other backend."""
    B, params, tokens, whole = _sample(monkeypatch, lambda T, old: T((10, 16), "f32", old.data[:160]), when)
    last = 5 if when == "release" else 12
    assert [pos for _, pos, _ in tokens] == list(range(5, last)) and whole == list(range(last + 1, 21))
    assert not any(n == 2 * 64 * 3 * 16 * 4 for n, _ in B.lib.blocks.values())          # the cache went back
