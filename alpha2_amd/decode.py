"""The logits behind a growing context, from kept keys and values.

Generation (packages/train/src/sample.ts:36-198) asks for the logits behind the last token of a context that grows by one token at
a time, and the reference runs the forward pass over all of it each time.  Where every row attends to the rows before it through
their keys and values alone (`attention == "heads"`, no dropout), those of earlier rows are what they were: the context is run once,
its q, k, v projections are kept, and a token after that costs one row (ah_decode).  Same arithmetic, other orders of summation."""
from __future__ import annotations

import ctypes as C
import math
from typing import Callable, Optional

import numpy as np

from . import _ffi as ffi
from ._ffi import check
from .autograd import Ctx, Tape
from .backend import HipBackend, TensorData
from .model import ModelConfig, ffn_dim, flashHeadSize, gptBlocks

# bases of the MLP activations, as HipBackend.CHANNEL_BASES numbers them, and the parameter that holds each one's coefficients
_ACTIVATIONS = {"gelu": {2: None}, "silu": {0: None}, "relu": {1: None}, "universal": {0: "act_gate", 3: "act_skip"},
                "kan_spline": {0: "kan_c0", 1: "kan_c1", 2: "kan_c2", 3: "kan_c3", 4: "kan_c4"}, "swiglu": {}}


class KeptContext:
    """Use `of`, then `lastRow` with a context that is one token longer each time, then `close`; `refresh` after code that may have moved
    a parameter.  The parameters' values must stay: the kept keys and values are not computed again."""

    @staticmethod
    def of(cfg: ModelConfig, params: dict, backend, longest: int) -> Optional["KeptContext"]:
        """None where the pass over the whole context has to stay: another backend or wiring of attention, sizes the kernels do not
        take, parameters of other shapes or types than the configuration's, or no memory for the keys and values."""
        act = cfg.ffnActivation or "gelu"
        if type(backend) is not HipBackend or cfg.attention != "heads" or cfg.dropout != 0 or act not in _ACTIVATIONS:
            return None
        width, ffn = cfg.nEmbd, ffn_dim(cfg)
        if width % cfg.nHead or not flashHeadSize(width // cfg.nHead) or width > 4096 or ffn % 4 or cfg.nLayer < 1 or len(params["layers"]) != cfg.nLayer:
            return None
        kept = KeptContext(cfg, params, backend, act, longest)
        try:
            if not kept._fits():
                return None
            # as many rows as the next power of two has: contexts of similar length ask the pool for blocks of one size
            kept.rows = min(cfg.blockSize, 1 << max(6, (longest - 1).bit_length()))
            kept.kv = backend._new((cfg.nLayer, kept.rows, 3 * width))
            kept.logits = backend._new((cfg.vocabSize,))
        except ffi.AlphaHipError:
            kept.close()
            return None
        except (KeyError, AttributeError):
            return None
        kept.describe()
        return kept

    def __init__(self, cfg: ModelConfig, params: dict, backend: HipBackend, act: str, longest: int):
        self.cfg, self.params, self.backend, self.act, self.longest = cfg, params, backend, act, longest
        self.kv: Optional[TensorData] = None
        self.logits: Optional[TensorData] = None
        self.rows = self.known = 0

    def _tensors(self):
        """Every parameter with the shape it must have; wpe may have more rows than are used."""
        cfg, p = self.cfg, self.params
        C_, V, F = cfg.nEmbd, cfg.vocabSize, ffn_dim(cfg)
        yield p["wte"].data, (V, C_)
        yield p["wpe"].data, (max(self.longest, p["wpe"].data.shape[0]), C_)
        for v in (p["lnF"]["weight"], p["lnF"]["bias"]):
            yield v.data, (C_,)
        yield p["lmHead"].data, (V, C_)
        for l in p["layers"]:
            for v in (l["ln1"]["weight"], l["ln1"]["bias"], l["ln2"]["weight"], l["ln2"]["bias"]):
                yield v.data, (C_,)
            m = l["mlp"]
            names = ("fc_gate", "fc_up", "fc_proj") if self.act == "swiglu" else ("fc1", "fc2")
            for v, shape in ((l["attn"]["wqkv"], (3 * C_, C_)), (l["attn"]["wo"], (C_, C_)), *((m[n], (F, C_)) for n in names[:-1]), (m[names[-1]], (C_, F))):
                yield v.data, shape
            for name in _ACTIVATIONS[self.act].values():
                if name is not None:
                    yield m[name].data, (1, F)

    def _fits(self) -> bool:
        return all(t.dtype == "f32" and t.store == "f32" and t.shape == shape and not self.backend._ptr(t) & 15 for t, shape in self._tensors())

    def refresh(self) -> bool:
        """After code of the caller's, which may have moved a parameter: False where one is no longer what the kernels take."""
        try:
            if not self._fits():
                return False
        except (ffi.AlphaHipError, KeyError, AttributeError):
            return False
        self.describe()
        return True

    def describe(self):
        """Where the parameters lie now."""
        cfg, p, ptr = self.cfg, self.params, self.backend._ptr
        bases = _ACTIVATIONS[self.act]
        gated = self.act == "swiglu"
        self.layers = (ffi.AhDecodeLayer * cfg.nLayer)()
        for out, l in zip(self.layers, p["layers"]):
            m = l["mlp"]
            out.ln1_w, out.ln1_b = ptr(l["ln1"]["weight"].data), ptr(l["ln1"]["bias"].data)
            out.wqkv, out.wo = ptr(l["attn"]["wqkv"].data), ptr(l["attn"]["wo"].data)
            out.ln2_w, out.ln2_b = ptr(l["ln2"]["weight"].data), ptr(l["ln2"]["bias"].data)
            out.fc1, out.up, out.fc2 = ((ptr(m["fc_gate"].data), ptr(m["fc_up"].data), ptr(m["fc_proj"].data)) if gated
                                        else (ptr(m["fc1"].data), 0, ptr(m["fc2"].data)))
            for k, name in bases.items():
                out.coef[k] = 0 if name is None else ptr(m[name].data)
        act = ffi.DECODE_GATED if gated else sum(1 << k for k in bases)
        cap = cfg.softCap if cfg.softCap is not None else 30.0
        self.model = ffi.AhDecode(cfg.vocabSize, cfg.nEmbd, cfg.nHead, ffn_dim(cfg), cfg.nLayer, act, self.rows,
                                  1 / math.sqrt(cfg.nEmbd // cfg.nHead), cap, 1e-5, ptr(p["wte"].data), ptr(p["wpe"].data),
                                  ptr(p["lnF"]["weight"].data), ptr(p["lnF"]["bias"].data), ptr(p["lmHead"].data), ptr(self.kv), ptr(self.logits))

    def lastRow(self, context: np.ndarray, releaseTensor: Optional[Callable]) -> np.ndarray:
        """Logits behind the last token of `context`: the context of the call before and one token, or, the first time, any."""
        lib, n = self.backend.lib, int(context.size)
        if not 0 < n <= min(self.longest, self.rows):           # past that, rows of the next layer would be overwritten
            raise ValueError(f"a context of {n} tokens, where 1 to {min(self.longest, self.rows)} were asked for")
        if self.known == n - 1 and self.known > 0:
            check(lib.ah_decode(C.byref(self.model), self.layers, int(context[-1]), n - 1))
        else:
            self._run(context, releaseTensor)
        self.known = n
        return self.backend._download(self.logits)

    def _run(self, context: np.ndarray, releaseTensor: Optional[Callable]):
        B, n, width = self.backend, int(context.size), self.cfg.nEmbd
        ids = TensorData((1, n), "i32", context.copy())
        tape = Tape()
        ctx = Ctx(tape, B, keptQkv=[])
        x = gptBlocks(ctx, self.cfg, self.params, ids)
        for i, qkv in enumerate(ctx.keptQkv):
            check(B.lib.ah_copy(B._ptr(self.kv) + i * self.rows * 3 * width * 4, B._ptr(qkv.data), n * 3 * width * 4))
        check(B.lib.ah_decode_head(C.byref(self.model), B._ptr(x.data) + (n - 1) * width * 4))
        tape.clear(releaseTensor)
        if releaseTensor is not None:
            releaseTensor(ids)

    def close(self):
        for t in (self.kv, self.logits):
            if t is not None:
                self.backend.releaseGpuTensor(t)
        self.kv = self.logits = None
