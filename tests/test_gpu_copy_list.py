"""ah_copy_list: several small copies and values in one launch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_copies_of_every_alignment_and_values_in_two_launches():
    """30 items (24 to a launch), offsets and lengths that allow 16, 4 or 1 byte at a time, values of 1 to 8 bytes, empty items; nothing
    beside the destinations changes."""
    from alpha2_amd import HipBackend, _ffi as ffi
    from alpha2_amd.backend import TensorData
    B = HipBackend(0)
    rs = np.random.RandomState(3)
    src = rs.randint(0, 256, 40000).astype(np.uint8)
    want = rs.randint(0, 256, 400000).astype(np.uint8)
    s, d = (TensorData((x.size // 4,), "i32", x.view(np.int32)) for x in (src, want))
    ps, pd = B._ptr(s), B._ptr(d)
    want = want.copy()
    items, at = [], 0
    for i, (a, b, n) in enumerate([(0, 0, 16384), (16, 32, 48), (4, 8, 20), (1, 3, 17), (0, 16, 15), (7, 0, 1), (0, 0, 0), (8, 4, 4096), (3, 5, 9000)] * 2):
        items.append(ffi.AhCopy(pd + at + a, ps + b, n, 0))
        want[at + a:at + a + n] = src[b:b + n]
        at += 16416
    for n in (1, 2, 3, 4, 5, 6, 7, 8, 8, 4, 1, 0):
        items.append(ffi.AhCopy(pd + at, 0, n, 0x8877665544332211))
        want[at:at + n] = np.frombuffer(np.uint64(0x8877665544332211).tobytes(), np.uint8)[:n]
        at += 16
    assert len(items) == 30
    ffi.check(B.lib.ah_copy_list((ffi.AhCopy * 30)(*items), 30))
    B._dirty(d)
    assert np.array_equal(d.data.view(np.uint8), want)
    for bad in (ffi.AhCopy(0, ps, 4, 0), ffi.AhCopy(pd, 0, 9, 0)):
        with pytest.raises(ffi.AlphaHipError):
            ffi.check(B.lib.ah_copy_list((ffi.AhCopy * 1)(bad), 1))
