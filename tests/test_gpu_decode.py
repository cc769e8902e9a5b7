"""Kept keys and values (ah_decode) against the same model in 64 bits, beside the pass over the whole context."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def B():
    from alpha2_amd import HipBackend
    return HipBackend(0)


def _model(B, vocab, ctx, layers, width, heads, **more):
    from alpha2_amd.model import ModelConfig, initGPT
    from alpha2_amd.rng import SeededRng
    cfg = ModelConfig(vocabSize=vocab, blockSize=ctx, nLayer=layers, nEmbd=width, nHead=heads, **more)
    params = initGPT(cfg, B, SeededRng(3))
    rs = np.random.RandomState(5)
    for l in params["layers"]:                  # gains, biases and coefficients that are not all the same
        for v in (l["ln1"]["weight"], l["ln1"]["bias"], l["ln2"]["weight"], l["ln2"]["bias"],
                  *(l["mlp"][n] for n in l["mlp"] if n.startswith(("act_", "kan_")))):
            v.data.data = v.data.data + 0.2 * rs.standard_normal(v.data.data.size).astype(np.float32)
        l["attn"]["wqkv"].data.data *= 75.0 / math.sqrt(width)      # q and k of 1.5, scores of a few units whatever the width: the softmax is not flat
    return cfg, params


def _logits64(cfg, params, tokens):
    """All rows' logits in 64 bits."""
    f = lambda v: v.data.data.reshape(v.data.shape).astype(np.float64)
    sigmoid = lambda x: 1 / (1 + np.exp(-x))
    silu = lambda x: x * sigmoid(x)
    gelu = lambda x: x * sigmoid(2 * math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3))

    def norm(x, p):
        c = x - x.mean(1, keepdims=True)
        return c / np.sqrt((c * c).mean(1, keepdims=True) + 1e-5) * f(p["weight"]) + f(p["bias"])
    T, H, C = len(tokens), cfg.nHead, cfg.nEmbd
    cap, act = 30.0 if cfg.softCap is None else cfg.softCap, cfg.ffnActivation
    x = f(params["wte"])[tokens] + f(params["wpe"])[:T]
    for l in params["layers"]:
        q, k, v = ((norm(x, l["ln1"]) @ f(l["attn"]["wqkv"]).T)[:, i * C:(i + 1) * C].reshape(T, H, C // H).transpose(1, 0, 2) for i in range(3))
        s = q @ k.transpose(0, 2, 1) / math.sqrt(C // H)
        if cap > 0:
            s = cap * np.tanh(s / cap)
        s = np.where(np.tril(np.ones((T, T), bool)), s, -np.inf)
        p = np.exp(s - s.max(2, keepdims=True))
        x = x + (p / p.sum(2, keepdims=True) @ v).transpose(1, 0, 2).reshape(T, C) @ f(l["attn"]["wo"]).T
        y, m = norm(x, l["ln2"]), l["mlp"]
        if act == "swiglu":
            x = x + (silu(y @ f(m["fc_gate"]).T) * (y @ f(m["fc_up"]).T)) @ f(m["fc_proj"]).T
            continue
        h = y @ f(m["fc1"]).T
        if act == "universal":
            h = silu(h) * f(m["act_gate"]) + h * f(m["act_skip"])
        elif act == "kan_spline":
            h = silu(h) * f(m["kan_c0"]) + np.maximum(h, 0) * f(m["kan_c1"]) + gelu(h) * f(m["kan_c2"]) + h * f(m["kan_c3"]) + h * h * f(m["kan_c4"])
        else:
            h = {"gelu": gelu, "silu": silu, "relu": lambda x: np.maximum(x, 0)}[act](h)
        x = x + h @ f(m["fc2"]).T
    return norm(x, params["lnF"]) @ f(params["lmHead"]).T


def _compare(kept, cfg, params, B, tokens, lengths, restart):
    """Both sum the same terms in fp32; the kept row sums its in shorter runs, so over the rows it is no further from 64 bits (root mean
    square of the rows' relative errors) than the pass over the whole context is, but for the scatter of a few dozen rows of which one
    ill-conditioned one weighs most: 1.5 times.  Where the sums are so short that both are single roundings away, the bound is those:
    eight after one another in a block (the norm's three, product, two on a score, exponential, weighted sum) and as many around the
    blocks, 2^-24 each."""
    from alpha2_amd.sample import _lastRow
    exact = _logits64(cfg, params, tokens)
    ours, theirs = [], []
    for n in lengths:
        if restart:
            kept.known = 0
            kept.lastRow(tokens[:n - 1], B.releaseGpuTensor)
        off = lambda row: np.linalg.norm(row.astype(np.float64) - exact[n - 1]) / np.linalg.norm(exact[n - 1])
        ours.append(off(kept.lastRow(tokens[:n], B.releaseGpuTensor)))
        theirs.append(off(_lastRow(cfg, params, B, tokens[:n], B.releaseGpuTensor)))
    ours, theirs = (math.sqrt(np.mean(np.square(e))) for e in (ours, theirs))
    print("off 64 bits: kept %.2e, whole context %.2e" % (ours, theirs))
    assert ours <= max(1.5 * theirs, 8 * (cfg.nLayer + 1) * 2.0 ** -24), (ours, theirs)


# widths on both sides of a lane's float4 counts (256, 512, 1024, 2048), head sizes of every group width and between two, rows of
# the head that fill no wave, every activation, with and without the cap
CASES = [
    (7, 80, 1, 8, 1, dict()),
    (97, 80, 2, 64, 4, dict(softCap=0.0)),
    (256, 80, 2, 256, 8, dict(ffnActivation="swiglu")),
    (2049, 40, 1, 264, 11, dict(ffnActivation="silu")),
    (300, 40, 1, 480, 6, dict(ffnActivation="universal")),
    (301, 40, 2, 768, 12, dict(ffnActivation="kan_spline")),
    (64, 24, 1, 1024, 8, dict(ffnActivation="relu")),
    (66, 24, 1, 1040, 13, dict(ffnDim=100)),
    (66, 24, 1, 2056, 257, dict(ffnDim=4100, ffnActivation="swiglu")),
]


@pytest.mark.parametrize("vocab,ctx,layers,width,heads,more", CASES)
def test_logits_behind_a_growing_context(B, vocab, ctx, layers, width, heads, more):
    from alpha2_amd.decode import KeptContext
    cfg, params = _model(B, vocab, ctx, layers, width, heads, **more)
    tokens = np.random.RandomState(1).randint(0, vocab, ctx).astype(np.int32)
    for prompt in (1, ctx // 2):
        kept = KeptContext.of(cfg, params, B, ctx)
        assert kept is not None
        _compare(kept, cfg, params, B, tokens, range(prompt, ctx + 1), False)
        kept.close()


@pytest.mark.parametrize("head_size", [16, 32, 64, 128])
def test_slices_of_a_long_context(B, head_size):
    """In one launch.  One key more than so many slices hold, and one less: 128 keys to a slice (64 and 32 of heads of 64 and 128 features), then, past 16
    of those, 16 longer ones."""
    from alpha2_amd.decode import KeptContext
    cfg, params = _model(B, 50, 2100, 1, 2 * head_size, 2)
    tokens = np.random.RandomState(2).randint(0, 50, 2100).astype(np.int32)
    kept, before = KeptContext.of(cfg, params, B, 2100), B.decodeStats()["oneLaunch"]
    lengths = (31, 32, 33, 62, 63, 64, 65, 127, 128, 129, 511, 512, 513, 577, 1023, 1024, 1025, 1026, 1199, 1200, 2047, 2048, 2049, 2100)
    _compare(kept, cfg, params, B, tokens, lengths, True)
    assert B.decodeStats()["oneLaunch"] - before == len(lengths)
    kept.close()


# every group width of the attention (and one between two), every count of float4s a lane of the joined row holds (1, 2, 3, 4, up to 8 and up to 16)
@pytest.mark.parametrize("width,heads,more", [
    (32, 2, dict(ffnDim=2052)), (64, 2, dict(ffnDim=2052)), (128, 2, dict(ffnDim=2052)), (256, 2, dict(ffnDim=2052)),
    (480, 6, dict(ffnDim=2052)), (768, 12, dict()), (1024, 64, dict(ffnDim=64)), (1152, 9, dict(ffnDim=64)), (2304, 18, dict(ffnDim=64)),
])
def test_slices_of_a_long_context_in_launches(B, width, heads, more):
    """64 keys to a slice up to 1024, then 16 longer ones; the slices are joined eight at a time."""
    from alpha2_amd.decode import KeptContext
    cfg, params = _model(B, 50, 1200, 1, width, heads, **more)
    tokens = np.random.RandomState(2).randint(0, 50, 1200).astype(np.int32)
    kept, before = KeptContext.of(cfg, params, B, 1200), B.decodeStats()["oneLaunch"]
    _compare(kept, cfg, params, B, tokens, (63, 64, 65, 128, 129, 512, 513, 577, 1024, 1025, 1026, 1200), True)
    assert B.decodeStats()["oneLaunch"] == before
    kept.close()


def test_what_the_kernels_do_not_take_runs_the_whole_context(B):
    from alpha2_amd import FastHipBackend
    from alpha2_amd.decode import KeptContext
    for more in (dict(attention="reference-flash"), dict(dropout=0.1), dict(ffnDim=6), dict(attention="unfused")):
        cfg, params = _model(B, 30, 16, 1, 32, 2, **more)
        assert KeptContext.of(cfg, params, B, 16) is None, more
    cfg, params = _model(B, 30, 16, 1, 40, 2)               # head size 20
    assert KeptContext.of(cfg, params, B, 16) is None
    cfg, params = _model(B, 30, 16, 1, 32, 2)
    assert KeptContext.of(cfg, params, FastHipBackend(0), 16) is None
    kept = KeptContext.of(cfg, params, B, 16)
    live = B.gpuMemStats()["liveAllocs"]
    kept.close()
    assert B.gpuMemStats()["liveAllocs"] == live - 2


def test_not_finite_parameters_reach_the_logits(B):
    from alpha2_amd.decode import KeptContext
    from alpha2_amd.sample import _lastRow
    cfg, params = _model(B, 30, 16, 1, 32, 2)
    params["wpe"].data.data[5 * 32] = np.nan                # position 5: seen from there on
    tokens = np.arange(8, dtype=np.int32)
    kept = KeptContext.of(cfg, params, B, 16)
    for n in range(1, 9):
        got, want = kept.lastRow(tokens[:n], B.releaseGpuTensor), _lastRow(cfg, params, B, tokens[:n], B.releaseGpuTensor)
        assert np.array_equal(np.isnan(got), np.isnan(want)), n
    kept.close()


@pytest.mark.parametrize("temperature", [0.0, 0.8])
@pytest.mark.parametrize("act", ["gelu", "swiglu"])
def test_the_same_tokens_with_and_without_kept_keys(B, monkeypatch, temperature, act):
    """Over a prompt of 60 and 20 tokens behind it, while flushGpu moves every parameter to another block and
    fills the one it left with NaN.  The largest logits lie further apart than the two ways' roundings put them (1e-4 of the row; see _compare)."""
    from alpha2_amd import sample
    from alpha2_amd.decode import KeptContext
    from alpha2_amd.model import collectParamEntries
    from alpha2_amd.rng import SeededRng
    cfg, params = _model(B, 50, 96, 2, 64, 4, ffnActivation=act)
    prompt = np.random.RandomState(4).randint(0, 50, 60)
    config = sample.SampleConfig(steps=20, temperature=temperature, topk=10)
    whole, gaps = [], []

    def look(row, *rest):
        top = np.sort(row)[::-1]
        gaps.append((top[0] - top[1]) / np.linalg.norm(row))
        return select(row, *rest)
    select = sample.selectToken
    with monkeypatch.context() as m:
        m.setattr(KeptContext, "of", staticmethod(lambda *a: None))
        if temperature == 0:
            m.setattr(sample, "selectToken", look)
        want = sample.sampleTokens(cfg, params, B, SeededRng(7), prompt, config, B.releaseGpuTensor, B.flush)
    assert not gaps or min(gaps) > 1e-4
    moved = {}

    def move():
        B.flush()
        for _, v in collectParamEntries(params):
            t = v.data
            t.data = np.array(t.data)
            old = t._buf.ptr
            B.releaseGpuTensor(t)
            for _ in range(1000):                       # (the pool hands out its lowest block first)
                x = B.full(t.shape, float("nan"))
                moved[x._buf.ptr] = x
                if x._buf.ptr == old:
                    break
            assert old in moved
        whole.append(1)
    got = sample.sampleTokens(cfg, params, B, SeededRng(7), prompt, config, B.releaseGpuTensor, move)
    assert len(whole) == 2 and got.size == 80 and np.array_equal(got, want)


# in one launch: an MLP that has more rows than q, k, v, one that has fewer than the residual stream, a head with more rows than the grid has waves, the
# widest model it takes (512, with rows of 2048), swiglu in pairs that fill no round, and one layer more than its arguments hold
CHAIN_CASES = [
    (5000, 40, 2, 64, 4, dict(ffnDim=2048)),
    (33, 40, 1, 256, 4, dict(ffnDim=36)),
    (260, 70, 2, 512, 4, dict()),
    (260, 40, 1, 512, 64, dict(ffnActivation="swiglu")),
    (64, 20, 33, 64, 2, dict()),
]


@pytest.mark.parametrize("vocab,ctx,layers,width,heads,more", CHAIN_CASES)
def test_a_token_in_one_launch(B, vocab, ctx, layers, width, heads, more):
    from alpha2_amd.decode import KeptContext
    cfg, params = _model(B, vocab, ctx, layers, width, heads, **more)
    tokens = np.random.RandomState(3).randint(0, vocab, ctx).astype(np.int32)
    kept, before = KeptContext.of(cfg, params, B, ctx), B.decodeStats()["oneLaunch"]
    _compare(kept, cfg, params, B, tokens, range(1, ctx + 1), False)
    assert B.decodeStats()["oneLaunch"] - before == (ctx - 1 if layers <= 32 else 0)
    kept.close()


@pytest.mark.parametrize("vocab,layers,width,heads,more,last", [
    (60, 2, 512, 4, dict(), 128), (60, 2, 272, 17, dict(), 512), (60, 2, 64, 2, dict(ffnDim=1028), 512), (60, 2, 256, 2, dict(), 1100),
    (2048, 1, 64, 2, dict(), 1100), (2049, 1, 64, 2, dict(), 0), (2049, 2, 64, 2, dict(), 1100),
])
def test_where_a_context_leaves_the_one_launch(B, vocab, layers, width, heads, more, last):
    """Past four slices of keys (32 to a slice for heads of 128 features, 128 for small ones) of a model wider than 256 or an MLP than 1024, and for one
    layer with a long head: the rows that a launch left are those the launches go on from."""
    from alpha2_amd.decode import KeptContext
    cfg, params = _model(B, vocab, 1100, layers, width, heads, **more)
    tokens = np.random.RandomState(4).randint(0, vocab, 1100).astype(np.int32)
    kept, before = KeptContext.of(cfg, params, B, 1100), B.decodeStats()["oneLaunch"]
    first = max(min(last, 1090) - 5, 20)
    kept.lastRow(tokens[:first - 1], B.releaseGpuTensor)
    _compare(kept, cfg, params, B, tokens, range(first, first + 12 if last < 1100 else 1101), False)
    taken = B.decodeStats()["oneLaunch"] - before
    assert taken == (0 if last == 0 else 6 if last < 1100 else 1101 - first), taken
    kept.close()


@pytest.mark.parametrize("width,heads,act", [(64, 2, "gelu"), (256, 8, "swiglu"), (512, 4, "kan_spline")])
def test_a_launch_that_gave_up_is_computed_again(B, width, heads, act):
    """Its waits end at the first word that is not there yet; the one workgroup behind it sums the same terms in the same order."""
    from alpha2_amd.decode import KeptContext
    cfg, params = _model(B, 70, 80, 2, width, heads, ffnActivation=act)
    tokens = np.random.RandomState(6).randint(0, 70, 80).astype(np.int32)
    kept = KeptContext.of(cfg, params, B, 80)
    rows, before = [], B.decodeStats()
    for given_up in (False, True):
        kept.known = 0
        kept.lastRow(tokens[:60], B.releaseGpuTensor)
        for n in range(61, 81):
            if given_up and n % 3 == 0:
                B.lib.ah_decode_next_ticks(-1)
            rows.append(kept.lastRow(tokens[:n], B.releaseGpuTensor).copy())
    after = B.decodeStats()
    assert after["oneLaunch"] - before["oneLaunch"] == 40 and after["computedAgain"] - before["computedAgain"] == 6
    for n, (a, b) in enumerate(zip(rows[:20], rows[20:])):
        assert np.array_equal(a, b), n + 61
    kept.close()


def test_a_computation_that_is_given_up_twice_is_seen(B):
    """Its logits are not those of the token before but NaN; the contexts behind it are computed as ever."""
    from alpha2_amd.decode import KeptContext
    cfg, params = _model(B, 70, 80, 2, 64, 2)
    tokens = np.random.RandomState(6).randint(0, 70, 80).astype(np.int32)
    kept = KeptContext.of(cfg, params, B, 80)
    kept.lastRow(tokens[:60], B.releaseGpuTensor)
    want = kept.lastRow(tokens[:61], B.releaseGpuTensor).copy()
    B.lib.ah_decode_next_ticks(-2)
    assert np.isnan(kept.lastRow(tokens[:62], B.releaseGpuTensor)).all()
    kept.known = 0
    kept.lastRow(tokens[:60], B.releaseGpuTensor)
    assert np.array_equal(kept.lastRow(tokens[:61], B.releaseGpuTensor), want)
    kept.close()


def test_the_end_of_waits_is_one_tokens(B):
    """Set for a token that takes the launches of a layer or is refused, it does not wait for a later one."""
    import ctypes

    from alpha2_amd.decode import KeptContext
    small, wide = (KeptContext.of(*_model(B, 40, 16, 1, width, heads), B, 16) for width, heads in ((64, 2), (576, 6)))
    tokens = np.arange(16, dtype=np.int32)
    for kept in (small, wide):
        kept.lastRow(tokens[:3], B.releaseGpuTensor)
    again = B.decodeStats()["computedAgain"]
    for token in (3, 4):
        B.lib.ah_decode_next_ticks(-1)
        if token == 3:
            wide.lastRow(tokens[:4], B.releaseGpuTensor)
        else:
            assert B.lib.ah_decode(ctypes.byref(small.model), small.layers, 99, 4) != 0
        small.lastRow(tokens[:token + 1], B.releaseGpuTensor)
    assert B.decodeStats()["computedAgain"] == again
    for kept in (small, wide):
        kept.close()


@pytest.mark.parametrize("layers,width,heads,act", [(2, 64, 8, "gelu"), (1, 256, 2, "swiglu"), (2, 512, 16, "silu"), (33, 64, 2, "gelu"), (2, 520, 5, "relu"), (1, 768, 12, "gelu")])
def test_the_first_token_reads_no_row_of_the_cache(B, layers, width, heads, act):
    """Position 0 on, in one launch and in launches, over a cache of NaN: rows 0 .. pos - 1 are read, and those are written before."""
    import ctypes

    from alpha2_amd import _ffi as ffi
    from alpha2_amd.decode import KeptContext
    from alpha2_amd.sample import _lastRow
    cfg, params = _model(B, 90, 70, layers, width, heads, ffnActivation=act)
    tokens = np.random.RandomState(8).randint(0, 90, 70).astype(np.int32)
    kept, exact = KeptContext.of(cfg, params, B, 70), _logits64(cfg, params, tokens)
    off = lambda row, n: np.linalg.norm(row.astype(np.float64) - exact[n]) / np.linalg.norm(exact[n])
    for count in (1, 2, 70):                     # (again from position 0, over what the run before has left behind it)
        ffi.check(B.lib.ah_fill_f32(kept.kv._buf.ptr, float("nan"), kept.kv.size))
        ours, theirs = [], []
        for n in range(count):
            ffi.check(B.lib.ah_decode(ctypes.byref(kept.model), kept.layers, int(tokens[n]), n))
            ours.append(off(B._download(kept.logits), n))
            theirs.append(off(_lastRow(cfg, params, B, tokens[:n + 1], B.releaseGpuTensor), n))
        ours, theirs = (math.sqrt(np.mean(np.square(e))) for e in (ours, theirs))
        assert ours <= max(1.5 * theirs, 8 * (cfg.nLayer + 1) * 2.0 ** -24), (count, ours, theirs)      # the bound of _compare
    kept.close()
