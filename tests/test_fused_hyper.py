"""What a fused step writes for the device's optimizer, on the CPU."""
import ctypes as C
import types

import numpy as np
import pytest

from alpha2_amd.fused import FusedTrainer
from alpha2_amd.train import TrainConfig


def _items(lr, seed, micro, drop=0.0, step=0):
    tc = TrainConfig(iters=10, lr=lr, lrMin=lr, warmupIters=-1, seed=seed)
    return FusedTrainer._hyper_items(types.SimpleNamespace(tc=tc, stepIdx=step, hyper=4096, drop=drop, seed_dev=8192, micro_steps=micro))


@pytest.mark.parametrize("lr", [3e-4, 1, 0.0, 1e-45, 3.4028235e38, 3.4028236e38, 1e39, float("inf")])
def test_the_learning_rate_is_what_a_32_bit_float_makes_of_it(lr):
    """Past the range, infinity."""
    (item,) = _items(lr, 0, 1)
    assert (item.dst, item.src, item.bytes) == (4096, 0, 4)
    with np.errstate(over="ignore"):
        assert item.value == int(np.float32(lr).view(np.uint32)) and C.c_float(lr).value == np.float32(lr)


def test_seeds_of_the_micro_steps():
    items = _items(1e-3, 2 ** 31 - 1, 3, drop=0.1, step=2)
    assert [(i.dst, i.bytes) for i in items[1:]] == [(8192, 4), (8196, 4), (8200, 4)]
    assert [i.value for i in items[1:]] == [(2 ** 31 - 1 + 2000 + m) % 2 ** 32 for m in range(3)]
