"""The work this library is measured on: whole training steps, evaluation passes, scoring passes and token sampling, through the
entry points a program uses (`FusedTrainer`, `Trainer` on `HipBackend` / `FastHipBackend`, `gptForward`, `sampleTokens`).

A case is a dict of plain values:
    do        "step"    one optimizer step (forward, backward, clip, update) on a batch it has not just seen
              "eval"    forward pass and mean loss of one batch cut from a device-resident corpus, the loss read back
              "score"   forward pass of one or a few ragged sequences, the logits left on the device (prefill)
              "sample"  token generation from a prompt, and the logits of the finished sequence
    how       "fused"   the hand-scheduled bf16 step in one hipGraph
              "fast"    the op interface with bf16 storage behind it; steps run under step plans
              "f32"     the op interface in fp32
    vocab, ctx, layers, width, heads, act, cap, attention, dropout     the model (cap < 0: the model's default)
    batch, tokens (per sequence), accum (micro-steps of a step), optimizer
    prompt, new, temperature                                            sampling only
Sizes are those of this repository's benchmark, tests and training-run tables, and draw() spreads over the range between them.
"""
import itertools
import math

import numpy as np
import torch
import torch.utils.checkpoint

from alpha2_amd import FastHipBackend, HipBackend, SeededRng
from alpha2_amd.autograd import Tape
from alpha2_amd.fused import FusedTrainer
from alpha2_amd.model import ModelConfig, collectParamEntries, ffn_dim, gptForward, initGPT
from alpha2_amd.sample import SampleConfig, sampleTokens
from alpha2_amd.train import DataLoader, TrainConfig, Trainer, zipfBatches


def _case(do, how, vocab, ctx, layers, width, heads, batch, **more):
    c = dict(do=do, how=how, vocab=vocab, ctx=ctx, layers=layers, width=width, heads=heads, batch=batch, tokens=ctx, accum=1,
             act="gelu", cap=-1.0, attention="heads", dropout=0.0, optimizer="adamw", prompt=0, new=0, temperature=0.0)
    c.update(more)
    return c


def listed():
    small = (50304, 1024, 12, 768, 12)
    return [
        # the smallest step anybody times: 2 layers x 128 at batch 2 x 64 (the reference's compiled-loop benchmark); all latency
        dict(_case("step", "fused", 256, 64, 2, 128, 4, 2), name="step-fused-2x128"),
        # a small model on a full batch with the regularisation and slab attention its training runs use (384 wide, 8 layers,
        # 512 tokens, batch 20): head size 48, rows that fill no power of two
        dict(_case("step", "fused", 4096, 512, 8, 384, 8, 20, attention="reference-flash", dropout=0.1), name="step-fused-8x384"),
        # the headline workload: the GPT-2-small-shape step, batch 16 x 1024
        dict(_case("step", "fused", *small, 16, attention="reference-flash"), name="step-fused-12x768"),
        # the large one: 350M parameters, four accumulated micro-steps of 8 x 1024
        dict(_case("step", "fused", 50304, 1024, 24, 1024, 16, 8, accum=4, attention="reference-flash"), name="step-fused-24x1024"),
        # the same headline step as an unchanged trainer issues it, op by op behind the interface, bf16 storage, step plans
        dict(_case("step", "fast", *small, 16), name="step-fast-12x768"),
        # parity mode: the tiny character-level model (4 layers x 128, batch 8 x 128), where launches and host work count
        dict(_case("step", "f32", 256, 128, 4, 128, 4, 8), name="step-f32-4x128"),
        # parity mode: the model and training defaults (6 layers x 256, 8 heads, batch 64 x 256)
        dict(_case("step", "f32", 256, 256, 6, 256, 8, 64), name="step-f32-6x256"),
        # parity mode: the GPT-2-small-shape step in fp32
        dict(_case("step", "f32", *small, 16), name="step-f32-12x768"),
        # validation loss of the default model on a batch that is a power of two in nothing
        dict(_case("eval", "f32", 256, 250, 6, 256, 8, 19, act="swiglu"), name="eval-f32-6x256"),
        # one long ragged sequence through the GPT-2-small shape in bf16: prefill
        dict(_case("score", "fast", *small, 1, tokens=777), name="score-fast-12x768"),
        # a sample from the default model as the trainer prints during training (64 tokens, temperature 0.8, top 40)
        dict(_case("sample", "f32", 256, 256, 6, 256, 8, 1, prompt=17, new=64, temperature=0.8), name="sample-f32-6x256"),
        # a continuation of a long prompt by the GPT-2-small shape, greedy
        dict(_case("sample", "f32", *small, 1, prompt=480, new=24), name="sample-f32-12x768"),
    ]


_LIMIT = {"fused": 1.5e13, "fast": 1e13, "f32": 6e12}          # operations of a drawn case, well under the listed ones' largest


def draw(rng):
    def spread(lo, hi):
        return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    do, how = rng.choice([("step", "fused")] * 4 + [("step", "fast"), ("step", "f32"), ("step", "f32"), ("eval", "f32"), ("eval", "fast"),
                                                    ("score", "f32"), ("score", "fast"), ("sample", "f32"), ("sample", "f32")])
    while True:
        vocab, ctx = spread(64, 50304), spread(32, 2048)
        layers = spread(1, 24 if how == "fused" or do != "step" else 10)
        heads, size = rng.randint(1, 16), rng.choice([16, 24, 32, 40, 48, 64, 64, 80, 96, 128])
        attention = rng.choice(["heads", "heads", "reference-flash"] if do == "sample" else ["heads", "reference-flash"])
        batch = spread(1, 64) if do in ("step", "eval") else rng.randint(1, 4) if do == "score" else 1
        if how == "fused":                                      # what the hand-scheduled step takes
            vocab = (vocab + 7) // 8 * 8
            unit = 128 if attention == "reference-flash" else 64
            heads = max(1, unit // size) * rng.randint(1, 12) if unit % size == 0 else 8 * rng.randint(1, 2)
        c = _case(do, how, vocab, ctx, layers, heads * size, heads, batch, attention=attention, cap=rng.choice([-1.0, -1.0, 0.0]),
                  act=rng.choice(["gelu", "gelu", "gelu", "swiglu", "silu", "universal", "kan_spline"]))
        if do == "step":
            c["accum"] = rng.choice([1, 1, 2, 4])
            c["optimizer"] = rng.choice(["adamw", "adamw", "adamw", "lion", "sgd"]) if how == "f32" else "adamw"
            c["dropout"] = rng.choice([0.0, 0.1]) if attention == "reference-flash" and how != "fast" else 0.0
        elif do == "score":
            c["tokens"] = rng.randint(ctx // 3, ctx)
        elif do == "sample":
            c["new"] = rng.randint(8, 48)
            c["prompt"] = rng.randint(1, ctx)
            c["temperature"] = rng.choice([0.0, 0.8])
        rows = c["batch"] * c["tokens"]
        if not 64 <= c["width"] <= 1024 or not (256 if attention == "reference-flash" else 16) <= rows <= 16384 or c["prompt"] + c["new"] > ctx:
            continue
        if how == "fused" and (c["width"] % unit or rows % 8):
            continue
        if _params(c) > 1.2e8 or _flops(c) > _LIMIT[how]:
            continue
        return c


# ---------------------------------------------------------------------------------------------- what a pass cannot do without
def _config(c):
    return ModelConfig(vocabSize=c["vocab"], blockSize=c["ctx"], nLayer=c["layers"], nEmbd=c["width"], nHead=c["heads"], dropout=c["dropout"],
                       ffnActivation=c["act"], softCap=None if c["cap"] < 0 else c["cap"], attention=c["attention"])


def _matrix_params(c):
    C, F = c["width"], ffn_dim(_config(c))
    return c["layers"] * (4 * C * C + (3 if c["act"] == "swiglu" else 2) * C * F) + c["vocab"] * C


def _params(c):
    return _matrix_params(c) + (c["vocab"] + c["ctx"]) * c["width"]


def _forward_flops(c, sequences, tokens):
    """Matrix products of every token, and the causal half of the score and value products."""
    return sequences * tokens * (2.0 * _matrix_params(c) + 2.0 * c["layers"] * c["width"] * tokens)


def _flops(c):
    if c["do"] == "step":
        return 3 * c["accum"] * _forward_flops(c, c["batch"], c["tokens"])
    if c["do"] == "sample":
        return 2 * _forward_flops(c, 1, c["prompt"] + c["new"])
    return _forward_flops(c, c["batch"], c["tokens"])


def work(case):
    P, rows = _params(case), case["batch"] * case["tokens"]
    if case["do"] == "step":
        # weights, gradients and both moments written, weights and moments read; the batch's ids
        nbytes = {"adamw": 28, "lion": 20, "sgd": 12}[case["optimizer"]] * P + 8 * rows * case["accum"]
    elif case["do"] == "sample":
        # one token depends on the one before: the weights are read for each, and once for the prompt and for the scores
        nbytes = 4 * (_matrix_params(case) * (case["new"] + 1) + (case["prompt"] + case["new"]) * (case["vocab"] + case["width"]))
    else:
        # the interface keeps f32 master weights; a matrix is read once in the type it is multiplied in, logits are written once
        size = 2 if case["how"] == "fast" else 4
        nbytes = size * (_matrix_params(case) + rows * case["vocab"]) + 8 * rows
    return {"bytes": float(nbytes), "flops": float(_flops(case))}


def tolerance(case):
    """Four times what other correct orders of summation show on these cases.  fp32: the fused attention against the same
    function op by op, two steps: gradients 3e-7 .. 8e-7, single values 1e-4 of a tensor's rms; an update whose sign is decided
    by a gradient of the size of that rounding moves one weight by twice the learning rate, 6e-3 of a weight's rms.  bf16: the
    hand-scheduled step against the op-by-op one, which round in other places: gradients 1e-3 .. 5e-3, rows of the token
    embedding that few tokens reach up to 0.5 of the tensor's rms; logits against fp32 1e-2.  fp32 with a vocabulary of 50304: the
head's gradient, 16384 terms summed one after the other, is 6.7e-5 from the 64-bit one where the other gradients are 1e-6."""
    if case["how"] == "f32":
        return {"rel": 3e-4 if case["do"] == "step" and case["vocab"] > 8192 else 1e-5, "max": 1e-2}
    return {"rel": 2e-2, "max": 0.9}


# ---------------------------------------------------------------------------------------------- inputs
class _Normal:
    """Initial weights: the generator `initGPT` draws from, on the GPU (the values are N(0, std) as with SeededRng)."""

    def __init__(self, seed):
        self.generator = torch.Generator(device="cuda").manual_seed(int(seed))

    def fillGauss(self, n, std):
        return torch.randn(n, generator=self.generator, device="cuda").mul_(std).cpu().numpy()


class _Memory:
    """Device memory of the library as torch sees foreign memory; keeps its owner alive."""

    def __init__(self, pointer, shape, kind, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": kind, "data": (pointer, False), "strides": None, "version": 3}


def _seen(pointer, shape, bf16=False, owner=None):
    t = torch.as_tensor(_Memory(pointer, shape, "<i2" if bf16 else "<f4", owner), device="cuda")
    return t.view(torch.bfloat16) if bf16 else t


def _tensor(backend, data):
    return _seen(backend._ptr(data), data.shape, data.store == "bf16", data)


_keys = itertools.count(1)


def _backend(case):
    backend = FastHipBackend(0) if case["how"] == "fast" else HipBackend(0)
    if backend.gpuMemStats()["bufferPoolBytes"] > 64 << 30:     # models of other sizes have been here: give their buffers back
        backend.purgeBufferPools()
    return backend


def _train_config(case):
    return TrainConfig(iters=200, batchSize=case["batch"], gradAccumSteps=case["accum"], optimizer=case["optimizer"])


def _batches(case, seed):
    """A ring of batches for four steps, cut from one stream of Zipf-distributed token ids."""
    return zipfBatches(seed % (1 << 30) + 1, 4 * case["accum"], case["batch"], case["tokens"], case["vocab"])


class _Fused:
    def __init__(self, case, seed):
        self.trainer = None
        backend, cfg = _backend(case), _config(case)
        self.trainer = FusedTrainer(backend, cfg, _train_config(case), case["batch"], accum=case["accum"],
                                    params=initGPT(cfg, backend, _Normal(seed)), index_in_step=True)
        self.ids = [self.trainer.add_batch(x, y) for x, y in _batches(case, seed)]
        self.accum, self.at = case["accum"], 0
        t = self.trainer
        self.out = {"loss": _seen(t.loss, (1,)), "weights": _seen(t.P, (t.nparam,)), "gradients": _seen(t.G, (t.nparam,))}

    def go(self):
        pick = [self.ids[(self.at + m) % len(self.ids)] for m in range(self.accum)]
        self.at += self.accum
        self.trainer.step(pick if self.accum > 1 else pick[0])
        return self.out

    def __del__(self):
        if self.trainer is not None:
            self.trainer.close()


class _Stepped:
    def __init__(self, case, seed):
        self.backend = backend = _backend(case)
        self.trainer = Trainer(backend, _config(case), _train_config(case), rng=_Normal(seed))
        self.batches = _batches(case, seed)
        for x, y in self.batches:
            backend.reshape(x, x.shape), backend.reshape(y, y.shape)            # resident before the first step
        self.accum, self.at, self.seen = case["accum"], 0, {}
        self.plan = next(_keys) if case["how"] == "fast" else 0

    def go(self):
        B, t = self.backend, self.trainer
        pick = [self.batches[(self.at + m) % len(self.batches)] for m in range(self.accum)]
        self.at += self.accum
        if self.plan:
            B.stepBegin(self.plan)
        r = t.step([(B.reshape(x, x.shape), B.reshape(y, y.shape)) for x, y in pick])
        if self.plan:
            B.stepEnd()
        # every matrix's gradient is in its first moment; a pass returns 64 tensors at most, so beside moments the weights are those
        # outside the layers
        moments = getattr(t.optimizer, "_m", {})
        matrices = [(n, v.data) for n, v in t.entries if len(v.data.shape) == 2 and v.data.shape[0] > 1]
        return {"loss": r.loss, "norm": r.gradNorm, "moments": self.look("moment", [(n, moments[n]) for n, _ in matrices if n in moments]),
                "weights": self.look("weight", [(n, d) for n, d in matrices if not moments or not n.startswith("layer.")])}

    def look(self, kind, named):
        out = {}
        for name, data in named:
            held = self.seen.get((kind, name))
            if held is None or held[0] is not data or held[1] != data._buf.ptr:
                held = self.seen[kind, name] = (data, data._buf.ptr, _tensor(self.backend, data))
            out[name] = held[2]
        return out

    def __del__(self):
        if getattr(self, "plan", 0):
            self.backend.resetStepPlan(self.plan)


class _Forward:
    """eval: batches from a corpus on the device, loss read back as evaluate() does.  score: ragged sequences, logits only."""

    def __init__(self, case, seed):
        self.backend, self.cfg = _backend(case), _config(case)
        self.params = initGPT(self.cfg, self.backend, _Normal(seed))
        length = case["batch"] * (case["tokens"] + 1) * 8
        (x, _), = zipfBatches(seed % (1 << 30) + 1, 1, 1, length, case["vocab"])
        self.loader = DataLoader(self.backend, x.data, SeededRng(seed % (1 << 30) + 7), case["batch"], case["tokens"])
        self.score = case["do"] == "score"

    def go(self):
        B = self.backend
        inputs, targets = self.loader.nextBatch()
        tape = Tape()
        r = gptForward(self.cfg, self.params, B, tape, inputs, None if self.score else targets)
        out = {"loss": 0.0 if self.score else float(r["loss"].data.data[0]), "logits": _tensor(B, r["logits"].data)}
        tape.clear(B.releaseGpuTensor, r["logits"])
        B.flush()
        return out


class _Sample:
    def __init__(self, case, seed):
        self.backend, self.cfg = _backend(case), _config(case)
        self.params = initGPT(self.cfg, self.backend, _Normal(seed))
        self.params["lmHead"].data.data *= 5.0                                  # logits spread as a trained model spreads them
        self.prompt = SeededRng(seed % (1 << 30) + 3).fillUniform(case["prompt"])
        self.prompt = np.floor(self.prompt * case["vocab"]).astype(np.int32)
        self.how = SampleConfig(steps=case["new"], temperature=case["temperature"], topk=40)
        self.seed = seed % (1 << 30) + 5

    def go(self):
        B = self.backend
        tokens = sampleTokens(self.cfg, self.params, B, SeededRng(self.seed), self.prompt, self.how, B.releaseGpuTensor, B.flush)
        tape = Tape()
        from_ids = B.fromArray(tokens, (1, len(tokens)), "i32")
        logits = gptForward(self.cfg, self.params, B, tape, from_ids)["logits"]
        out = {"tokens": tokens, "logits": _tensor(B, logits.data)}
        tape.clear(B.releaseGpuTensor, logits)
        return out


def prepare(case, seed):
    kind = {"eval": _Forward, "score": _Forward, "sample": _Sample}.get(case["do"]) or (_Fused if case["how"] == "fused" else _Stepped)
    return kind(case, seed)


def run(state):
    return state.go()


# ---------------------------------------------------------------------------------------------- the same passes in 64 bits
def _act64(case, h, p):
    """h: pre-activation (swiglu: gate and up); p(name): a parameter of the layer's MLP."""
    F, act = torch.nn.functional, case["act"]
    if act == "swiglu":
        return F.silu(h[0]) * h[1]
    if act == "silu":
        return F.silu(h)
    if act == "universal":
        return F.silu(h) * p("act_gate") + h * p("act_skip")
    gelu = F.gelu(h, approximate="tanh")
    if act == "kan_spline":
        return F.silu(h) * p("kan_c0") + F.relu(h) * p("kan_c1") + gelu * p("kan_c2") + h * p("kan_c3") + h * h * p("kan_c4")
    return gelu


def _block64(case, p, x):
    F, (B, T, C), H = torch.nn.functional, x.shape, case["heads"]
    D, cap = C // H, 30.0 if case["cap"] < 0 else case["cap"]
    qkv = F.layer_norm(x, (C,), p("ln1.weight"), p("ln1.bias"), 1e-5) @ p("attn.wqkv").t()
    if case["attention"] == "heads":
        q, k, v = (t.reshape(B, T, H, D).transpose(1, 2).contiguous() for t in qkv.split(C, 2))
    else:                                                       # the rows of a matrix re-read as slabs, no head transpose
        q, k, v = (t.reshape(B, H, T, D) for t in qkv.split(C, 2))
    s = q @ k.transpose(2, 3).contiguous() / math.sqrt(D)
    if cap > 0:
        s = cap * torch.tanh(s / cap)
    s = s.masked_fill(torch.ones(T, T, dtype=torch.bool, device=x.device).triu(1), -math.inf)
    x = x + (torch.softmax(s, 3) @ v).transpose(1, 2).reshape(B, T, C) @ p("attn.wo").t()
    y = F.layer_norm(x, (C,), p("ln2.weight"), p("ln2.bias"), 1e-5)
    if case["act"] == "swiglu":
        return x + _act64(case, (y @ p("mlp.fc_gate").t(), y @ p("mlp.fc_up").t()), None) @ p("mlp.fc_proj").t()
    return x + _act64(case, y @ p("mlp.fc1").t(), lambda n: p("mlp." + n)) @ p("mlp.fc2").t()


def _logits64(case, w, ids):
    x = w["wte"][ids] + w["wpe"][: ids.shape[1]]
    for l in range(case["layers"]):
        block = lambda x, l=l: _block64(case, lambda n: w["layer.%d.%s" % (l, n)], x)
        x = torch.utils.checkpoint.checkpoint(block, x, use_reentrant=False) if torch.is_grad_enabled() else block(x)
    return torch.nn.functional.layer_norm(x, (case["width"],), w["lnF.weight"], w["lnF.bias"], 1e-5) @ w["lmHead"].t()


def _loss64(logits, targets):
    return torch.nn.functional.cross_entropy(logits.reshape(-1, logits.shape[-1]), targets.reshape(-1))


def _ids(t):
    return torch.from_numpy(np.array(t.data, dtype=np.int64).reshape(t.shape)).cuda()


def _step64(case, seed, w):
    tc, names = _train_config(case), list(w)
    bare = {"wte", "wpe"} | {n for n in names if ".ln" in n or n.startswith("lnF")}                 # not decayed
    for t in w.values():
        t.requires_grad_(True)
    loss = 0.0
    for x, y in _batches(case, seed)[: case["accum"]]:
        part = _loss64(_logits64(case, w, _ids(x)), _ids(y))
        part.backward()
        loss += float(part.detach()) / case["accum"]
        del part
    norm = math.sqrt(sum(float((t.grad ** 2).sum()) for t in w.values())) / case["accum"]
    scale = min(1.0, tc.gradClip / norm) / case["accum"]
    low = tc.lr / 10                                            # the first step of the warm-up
    lr = low + (tc.lr - low) / min(2000, tc.iters // 5)
    grads, moments, after = {n: t.grad for n, t in w.items()}, {}, {}
    for n, t in w.items():
        t, g = t.detach(), grads[n] * scale
        if case["optimizer"] == "sgd":
            after[n] = t - lr * g
            continue
        decayed = t if n in bare else t * (1 - lr * tc.weightDecay)
        if case["optimizer"] == "lion":
            moments[n], after[n] = (1 - tc.beta2) * g, decayed - lr * torch.sign(g)
        else:
            moments[n], after[n] = (1 - tc.beta1) * g, decayed - lr * g / (g.abs() + tc.eps)
    if case["how"] == "fused":                                  # one arena: decayed, then not; every tensor from a multiple of 64 on
        order = [n for n in names if n not in bare] + [n for n in names if n in bare]
        flat = lambda d: torch.cat([torch.nn.functional.pad(d[n].reshape(-1), (0, -d[n].numel() % 64)) for n in order])
        return {"loss": torch.tensor([loss], dtype=torch.float64), "weights": flat(after), "gradients": flat(grads)}
    matrices = [n for n in names if w[n].ndim == 2 and w[n].shape[0] > 1]
    return {"loss": loss, "norm": norm, "moments": {n: moments[n] for n in matrices if moments},
            "weights": {n: after[n] for n in matrices if not moments or not n.startswith("layer.")}}


def _sample64(case, seed, w):
    rng = SeededRng(seed % (1 << 30) + 3)
    tokens = [int(t) for t in np.floor(rng.fillUniform(case["prompt"]) * case["vocab"])]
    rng = SeededRng(seed % (1 << 30) + 5)
    for _ in range(case["new"]):
        row = _logits64(case, w, torch.tensor([tokens], device="cuda"))[0, -1]
        if case["temperature"] <= 0:
            tokens.append(int(row.argmax()))
            continue
        row = row / case["temperature"]
        if case["vocab"] > 40:
            row = row.masked_fill(row < row.topk(40).values[-1], -math.inf)
        at = int((torch.softmax(row, 0).cumsum(0) <= rng.next()).sum())
        tokens.append(at if at < case["vocab"] else 0)
    return {"tokens": np.array(tokens, dtype=np.int32), "logits": _logits64(case, w, torch.tensor([tokens], device="cuda"))}


def exact(case, seed):
    """What the first run(prepare(case, seed)) returns, in 64 bits; None where masks of the library's own generator are in it."""
    if case["dropout"] > 0:
        return None
    w = {n: torch.from_numpy(v.data.data.reshape(v.data.shape)).cuda().double() for n, v in collectParamEntries(initGPT(_config(case), None, _Normal(seed)))}
    if case["do"] == "step":
        return _step64(case, seed, w)
    with torch.no_grad():
        if case["do"] == "sample":
            w["lmHead"] *= 5.0
            return _sample64(case, seed, w)
        length, T = case["batch"] * (case["tokens"] + 1) * 8, case["tokens"]
        (x, _), = zipfBatches(seed % (1 << 30) + 1, 1, 1, length, case["vocab"])
        corpus, rng = _ids(x).reshape(-1), SeededRng(seed % (1 << 30) + 7)
        starts = [math.floor(rng.next() * (length - T)) for _ in range(case["batch"])]
        cut = lambda by: torch.stack([corpus[s + by: s + by + T] for s in starts])
        logits = _logits64(case, w, cut(0))
        return {"loss": float(_loss64(logits, cut(1))) if case["do"] == "eval" else 0.0, "logits": logits}
