"""A pass of AdamW in tables (HipBackend.adamwSteps) against the tensors one by one, on the CPU: the backend's bookkeeping over a stand-in
for the native library whose device memory is host memory.  A freed block goes to the next request of its size, as from the device's pool, and
the tensors of a launch are updated last to first: on the device they run at the same time, so no result may hang on their order."""
import ctypes as C

import numpy as np
import pytest

from alpha2_amd import _ffi as ffi

HYPER = (1e-3, 0.9, 0.95, 1e-8, 0.1, 0.05)


class HostLibrary:
    """p += g, m += 1, v += 2 stands for the update: what is checked is which bytes meet, not the arithmetic."""

    def __init__(self):
        self.blocks, self.free, self.launches = {}, {}, []

    def ah_init(self, device):
        return 0

    def ah_alloc(self, nbytes, out):
        size = (int(nbytes) + 511) & ~511
        if self.free.get(size):
            address = self.free[size].pop()
        else:
            block = C.create_string_buffer(size)
            address = C.addressof(block)
            self.blocks[address] = (size, block)
        out._obj.value = address
        return 0

    def ah_free(self, address):
        assert all(address not in f for f in self.free.values())
        self.free.setdefault(self.blocks[address][0], []).append(address)
        return 0

    def ah_copy(self, dst, src, nbytes):
        C.memmove(dst, src, nbytes)
        return 0

    def ah_upload(self, dst, host, nbytes):
        C.memmove(dst, host, nbytes)
        return 0

    def ah_download(self, host, src, nbytes):
        C.memmove(host, src, nbytes)
        return 0

    def update(self, p, g, m, v, n):
        at = lambda address: np.frombuffer((C.c_char * (4 * n)).from_address(address), np.float32)
        at(p)[:] += at(g)
        at(m)[:] += 1
        at(v)[:] += 2

    def ah_adamw(self, p, g, m, v, n, *rest):
        self.launches.append(1)
        self.update(p, g, m, v, n)
        return 0

    def ah_adamw_list(self, items, count, *rest):
        self.launches.append(count)
        for q in reversed(items[:count]):
            self.update(q.p, q.g, q.m, q.v, q.n)
        return 0


@pytest.fixture
def B(monkeypatch):
    from alpha2_amd import HipBackend
    lib = HostLibrary()
    monkeypatch.setattr(ffi, "load", lambda: lib)
    return HipBackend(0)


def _tensor(seed, n=12):
    from alpha2_amd.backend import TensorData
    return TensorData((n,), "f32", np.random.RandomState(seed).randint(1, 100, n).astype(np.float32))


def _items(count):
    return [tuple(_tensor(4 * i + k) for k in range(4)) + (0.0,) for i in range(count)]


def _results(items):
    return [np.array(t.data) for row in items for t in row[:4]]


def _same(B, make):
    """make(): the items, made anew for each way."""
    one, many = make(), make()
    for p, g, m, v, wd in one:
        B.adamwStep(p, g, m, v, *HYPER[:4], wd, *HYPER[4:])
    B.lib.launches.clear()
    B.adamwSteps(many, *HYPER)
    assert all(np.array_equal(a, b) for a, b in zip(_results(one), _results(many)))
    return B.lib.launches


@pytest.mark.parametrize("count", [1, 8, 9, 60])
def test_tensors_of_their_own_share_launches(B, count):
    assert _same(B, lambda: _items(count)) == [n for n in (min(count, 8), min(count - 8, 48), count - 56) if n > 0]


@pytest.mark.parametrize("reader,writer", [(0, 1), (0, 3), (2, 0)])
@pytest.mark.parametrize("role", [0, 2, 3])
def test_a_gradient_that_another_item_updates(B, reader, writer, role):
    """As the parameter or a moment, before and after it is read."""
    def make():
        items = [list(row) for row in _items(4)]
        items[writer][role] = items[reader][1]
        return items
    _same(B, make)


@pytest.mark.parametrize("reader,writer", [(0, 1), (1, 0)])
@pytest.mark.parametrize("host", [False, True])
def test_a_gradient_that_overlaps_what_another_item_updates(B, reader, writer, host):
    """Views of one buffer that begin at different elements; host: the view has contents on the host that are still to be uploaded."""
    def make():
        items = [list(row) for row in _items(2)]
        whole = _tensor(99, 16)
        items[reader][1], items[writer][0] = B._view(whole, (12,)), B._view(whole, (12,), 16)
        if host:
            items[reader][1].data = np.arange(12)
        return items
    _same(B, make)


def test_a_gradient_and_a_parameter_that_are_views_of_a_clone(B):
    """The writer's view moves to a block of its own, and the gradient with it."""
    def make():
        items = [list(row) for row in _items(3)]
        whole = _tensor(98)
        make.clones.append(B.clone(whole))
        items[0][1], items[2][0] = B._view(whole, (12,)), whole
        return items
    make.clones = []
    _same(B, make)
    for c in make.clones:
        assert np.array_equal(c.data, _tensor(98).data)


@pytest.mark.parametrize("count", [3, 12])
def test_gradients_that_are_made_on_the_way(B, count):
    """Nobody else holds them: each block is free again as soon as the next one is asked for."""
    one, many = _items(count), _items(count)
    gradients = lambda rows: ((p, _tensor(1000 + i), m, v, wd) for i, (p, _, m, v, wd) in enumerate(rows))
    for p, g, m, v, wd in gradients(one):
        B.adamwStep(p, g, m, v, *HYPER[:4], wd, *HYPER[4:])
    B.adamwSteps(gradients(many), *HYPER)
    assert all(np.array_equal(a, b) for a, b in zip(_results(one), _results(many)))


def test_gradients_that_are_made_from_updated_parameters(B):
    """Items from an iterator: each one's update is done when the next is made."""
    from alpha2_amd.backend import TensorData

    def chain(rows):
        last = np.ones(12, np.float32)
        for p, _, m, v, wd in rows:
            yield p, TensorData((12,), "f32", last), m, v, wd
            last = np.array(p.data)
    one, many = _items(5), _items(5)
    for p, g, m, v, wd in chain(one):
        B.adamwStep(p, g, m, v, *HYPER[:4], wd, *HYPER[4:])
    B.adamwSteps(chain(many), *HYPER)
    assert all(np.array_equal(a, b) for a, b in zip(_results(one), _results(many)))


def test_an_optimizer_whose_gradient_is_a_later_parameter(B):
    """AdamW.step in the order of its parameters."""
    from alpha2_amd.train import AdamW

    def run(backend_steps):
        if not backend_steps:
            B.adamwStep = lambda *a: type(B).adamwStep(B, *a)           # an update of its own: one by one
        try:
            a, b, g = _tensor(1), _tensor(2), _tensor(3)
            AdamW(B).step({"a": a, "b": b}, {"a": b, "b": g})
            return np.array(a.data), np.array(b.data)
        finally:
            B.__dict__.pop("adamwStep", None)
    for x, y in zip(run(False), run(True)):
        assert np.array_equal(x, y)
