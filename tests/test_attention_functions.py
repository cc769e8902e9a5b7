"""tanh and exp of the fp32 attention's scores, value by value: the constants on the CPU, what the device makes of them through the calls
that return them whole."""
import ctypes as C
import math
import os
import re

import numpy as np
import pytest

SOURCE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "alpha2_amd", "csrc", "attention.hip")


def _constants():
    """The coefficients of tanh_small from the highest, its end, and the two parts of log2 e, as the source has them."""
    text = open(SOURCE).read()
    body = re.search(r"float tanh_small\(float x\) \{(.*?)\n\}", text, re.S).group(1)
    coefficients = [float(c) for c in re.findall(r"(-?\d\.\d+)f", body)]
    end, high, low = re.search(r"TANH_SMALL = ([\d.]+)f, LOG2E = ([\d.]+)f, LOG2E_REST = ([\d.e-]+)f", text).groups()
    return [float(np.float32(c)) for c in coefficients], float(end), float(np.float32(high)), float(np.float32(low))


def _off(got, want):
    """Distance in last places of the 32-bit number nearest to `want`."""
    return np.abs(got.astype(np.float64) - want) / np.spacing(np.abs(want).astype(np.float32)).astype(np.float64)


def test_the_polynomial_of_tanh():
    """x + x^3 P(x^2) with exact arithmetic: 0.15 of 2^-24 of the value at most; and no polynomial of that order is much
    better, as a fit of its own by reweighted least squares (Lawson) shows."""
    c, end, _, _ = _constants()
    assert len(c) == 5
    x = end * (0.5 - 0.5 * np.cos(np.linspace(1e-3, math.pi, 4001)))
    error = lambda c: x + x ** 3 * np.polyval(c, x * x) - np.tanh(x)
    relative = lambda c: np.abs(error(c) / np.tanh(x))
    assert relative(c).max() <= 0.15 * 2.0 ** -24, relative(c).max() * 2 ** 24
    weight = np.ones_like(x)
    columns = np.stack([x ** (3 + 2 * k) / np.tanh(x) for k in range(4, -1, -1)], 1)
    best = np.inf
    for _ in range(200):
        w = np.sqrt(weight)[:, None]
        fit = np.linalg.lstsq(columns * w, ((np.tanh(x) - x) / np.tanh(x))[:, None] * w, rcond=None)[0][:, 0]
        r = relative(fit)
        best = min(best, r.max())
        weight *= r / r.mean()
        weight /= weight.mean()
    assert relative(c).max() <= 3 * best, (relative(c).max(), best)        # (the coefficients are 32-bit numbers, the fit's are not)


def test_the_two_parts_of_log2_e():
    """Together right to 2^-24 of the second; the first is the nearest 32-bit number."""
    _, _, high, low = _constants()
    assert high == float(np.float32(1 / math.log(2)))
    assert abs(high + low - 1 / math.log(2)) <= 2.0 ** -24 * low


# ---------------------------------------------------------------------------------------------- on the device
@pytest.fixture(scope="module")
def B():
    from alpha2_amd import HipBackend
    return HipBackend(0)


HEADS = 65535


def _flash(B, q, k, v, o, g, lse, cap, backward):
    """One position a head, head size 8: heads of [q, 0 ..], [k, 0 ..], ..; returns what is left in lse and the first feature of dV."""
    from alpha2_amd import _ffi as ffi
    from alpha2_amd.backend import TensorData

    def wide(x):
        w = np.zeros((HEADS, 8), np.float32)
        w[:, 0] = x
        return TensorData(w.shape, "f32", w)
    t = [wide(x) for x in (q, k, v, o, g)]
    l = TensorData((HEADS,), "f32", np.asarray(lse, np.float32) * np.ones(HEADS, np.float32))
    d = [B._new((HEADS, 8)) for _ in range(3)]
    st = (HEADS * 8, 8, 8)
    p = [B._ptr(x) for x in (*t, l)]
    f = ffi.AhFlash(ffi.F32, 1, HEADS, 1, 8, *st, *st, *st, *st, 1.0, cap, *p[:4], p[5], p[4], *(x._buf.ptr for x in d), 0, 0)
    ffi.check((B.lib.ah_flash_bwd if backward else B.lib.ah_flash_fwd)(C.byref(f)))
    return B._download(l), d[2].data.reshape(HEADS, 8)[:, 0]


@pytest.mark.gpu
def test_tanh_of_every_size(B):
    """A single key weighs 1, so the logarithm of the weights' sum is its score: tanh of q k under a cap of 1.  0.73 last places at most below
    0.625, 1.63 from there on, as stated beside the functions (measured over every value from 0.5 to 1, where both are worst); odd, and
    1 where the exponential overflows."""
    rng = np.random.default_rng(0)
    at = int(np.float32(0.625).view(np.uint32))
    for bound, make in ((0.73, lambda: 2.0 ** rng.uniform(-12, math.log2(0.625), HEADS)),
                        (0.73, lambda: np.arange(at - HEADS, at, dtype=np.uint32).view(np.float32)), (1.63, lambda: np.arange(at, at + HEADS, dtype=np.uint32).view(np.float32)),
                        (1.63, lambda: rng.uniform(0.625, 1, HEADS)), (1.63, lambda: rng.uniform(0.625, 10, HEADS)), (1.63, lambda: 2.0 ** rng.uniform(3, 100, HEADS))):
        for _ in range(4):
            x = (make() * rng.choice([-1, 1], HEADS)).astype(np.float32)
            got, _ = _flash(B, x, 1, 0, 0, 0, 0, 1.0, False)
            assert _off(got, np.tanh(x.astype(np.float64))).max() <= bound


@pytest.mark.gpu
def test_exp_of_every_size(B):
    """The weight of a single key whose score is zero is exp(-lse), lse as the caller gives it, and dV is that weight times a gradient of 1:
    0.96 last places off at most; nothing below the range."""
    rng = np.random.default_rng(1)
    worst = 0
    for low, high in ((-1, 0.01), (-20, 0), (-87, 0), (-1e-3, 0)):
        for _ in range(8):
            x = rng.uniform(low, high, HEADS).astype(np.float32)
            _, got = _flash(B, 0, 0, 0, 0, 1, -x, 0.0, True)
            worst = max(worst, _off(got, np.exp(x.astype(np.float64))).max())
    assert worst <= 0.96
    x = -np.float32(2) ** rng.uniform(7.4, 29, HEADS).astype(np.float32)             # past the smallest number
    assert not _flash(B, 0, 0, 0, 0, 1, -x, 0.0, True)[1].any()
