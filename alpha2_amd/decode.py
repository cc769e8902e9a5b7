"""The logits behind a growing context, from kept keys and values.

Generation (packages/train/src/sample.ts:36-198) asks for the logits behind the last token of a context that grows by one token at
a time, and the reference runs the forward pass over all of it each time.  Where every row attends to the rows before it through
their keys and values alone (`attention == "heads"`, no dropout), those of earlier rows are what they were: the context is run once,
its q, k, v projections are kept, and a token after that costs one row (ah_decode).  Same arithmetic, other orders of summation."""
from __future__ import annotations

import ctypes
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


def mayMove(callback: Optional[Callable]) -> bool:
    """Is this code of the caller's own, which may move a parameter?  The backend's release and flush move none, and a look at all
    parameters after each is 1.6 % of sampling 24 tokens from the GPT-2-small shape."""
    return callback is not None and getattr(callback, "__func__", None) not in (HipBackend.releaseGpuTensor, HipBackend.flush)


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
        if not kept.refresh():
            return None
        try:
            # as many rows as the next power of two has: contexts of similar length ask the pool for blocks of one size
            kept.rows = min(cfg.blockSize, 1 << max(6, (longest - 1).bit_length()))
            kept.kv = backend._new((cfg.nLayer, kept.rows, 3 * width))
            kept.logits = backend._new((cfg.vocabSize,))
        except ffi.AlphaHipError:
            kept.close()
            return None
        kept.model.rows, kept.model.kv, kept.model.logits = kept.rows, kept.kv._buf.ptr, kept.logits._buf.ptr
        return kept

    def __init__(self, cfg: ModelConfig, params: dict, backend: HipBackend, act: str, longest: int):
        self.cfg, self.params, self.backend, self.longest = cfg, params, backend, longest
        self.kv: Optional[TensorData] = None
        self.logits: Optional[TensorData] = None
        self.rows = self.known = 0
        bases, C_, F = _ACTIVATIONS[act], cfg.nEmbd, ffn_dim(cfg)
        self.act = ffi.DECODE_GATED if act == "swiglu" else sum(1 << k for k in bases)
        # the MLP's parameters by name (None: there is none), and the shapes of _parameters ((): none, None: wpe's)
        self.mlp = (("fc_gate", "fc_up", "fc_proj") if act == "swiglu" else ("fc1", None, "fc2")) + tuple(bases.get(k) for k in range(5))
        self.shapes = cfg.nLayer * [(C_,), (C_,), (3 * C_, C_), (C_, C_), (C_,), (C_,), (F, C_), (F, C_) if act == "swiglu" else (), (C_, F),
                                    *((1, F) if bases.get(k) else () for k in range(5))]
        self.shapes += [(cfg.vocabSize, C_), None, (C_,), (C_,), (cfg.vocabSize, C_)]

    def _parameters(self):
        """The tensors of AhDecodeLayer's fields, layer by layer, then those of AhDecode."""
        p, (gate, up, down, *coefs) = self.params, self.mlp
        for l in p["layers"]:
            ln1, ln2, attn, m = l["ln1"], l["ln2"], l["attn"], l["mlp"]
            yield from (ln1["weight"].data, ln1["bias"].data, attn["wqkv"].data, attn["wo"].data, ln2["weight"].data, ln2["bias"].data,
                        m[gate].data, up and m[up].data, m[down].data)
            for name in coefs:
                yield name and m[name].data
        yield from (p["wte"].data, p["wpe"].data, p["lnF"]["weight"].data, p["lnF"]["bias"].data, p["lmHead"].data)

    def refresh(self) -> bool:
        """Where the parameters lie now (again after code of the caller's, which may have moved one); False where one is not what the
        kernels take."""
        cfg, ptr = self.cfg, self.backend._ptr
        at = []
        try:
            wpe = self.params["wpe"].data.shape             # may have more rows than are used
            for t, shape in zip(self._parameters(), self.shapes):
                if shape == ():
                    at.append(0)
                elif t.shape == (shape or (max(self.longest, wpe[0]), cfg.nEmbd)) and t.dtype == "f32" and t.store == "f32":
                    at.append(ptr(t))
                else:
                    return False
        except (ffi.AlphaHipError, KeyError, AttributeError):
            return False
        if any(map((15).__and__, at)):
            return False
        self.layers = (ffi.AhDecodeLayer * cfg.nLayer).from_buffer((ctypes.c_uint64 * len(at))(*at))
        cap = cfg.softCap if cfg.softCap is not None else 30.0
        kv, logits = (0 if t is None else t._buf.ptr for t in (self.kv, self.logits))
        self.model = ffi.AhDecode(cfg.vocabSize, cfg.nEmbd, cfg.nHead, ffn_dim(cfg), cfg.nLayer, self.act, self.rows,
                                  1 / math.sqrt(cfg.nEmbd // cfg.nHead), cap, 1e-5, *at[-5:], kv, logits)
        return True

    def lastRow(self, context: np.ndarray, releaseTensor: Optional[Callable]) -> np.ndarray:
        """Logits behind the last token of `context`: the context of the call before and one token, or, the first time, any."""
        lib, n = self.backend.lib, int(context.size)
        if not 0 < n <= min(self.longest, self.rows):           # past that, rows of the next layer would be overwritten
            raise ValueError(f"a context of {n} tokens, where 1 to {min(self.longest, self.rows)} were asked for")
        if self.known == n - 1 and self.known > 0:
            check(lib.ah_decode(ctypes.byref(self.model), self.layers, int(context[-1]), n - 1))
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
        check(B.lib.ah_decode_head(ctypes.byref(self.model), B._ptr(x.data) + (n - 1) * width * 4))
        tape.clear(releaseTensor)
        if releaseTensor is not None:
            releaseTensor(ids)

    def close(self):
        for t in (self.kv, self.logits):
            if t is not None:
                self.backend.releaseGpuTensor(t)
        self.kv = self.logits = None
