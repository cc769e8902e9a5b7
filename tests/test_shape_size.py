"""The number of elements of a shape, whatever its extents are counted in."""
import numpy as np
import pytest

from alpha2_amd.backend import TensorData, shapeSize


@pytest.mark.parametrize("kind", [int, np.int16, np.int32, np.uint32, np.int64])
def test_elements_past_the_type_of_the_extents(kind):
    """2^14 four times, 300 three times: past 32 and 16 bits."""
    wide = [kind(1 << 14)] * 4
    assert shapeSize(wide) == 1 << 56 and type(shapeSize(wide)) is int
    assert shapeSize((kind(300), kind(300))) == 90000
    assert shapeSize(np.array([300, 300, 300], kind)) == 27000000


def test_extents_are_cut_to_whole_numbers_one_by_one():
    """As a tensor of that shape has them."""
    for shape in ((2.5, 3.5), (), (0, 7), ("3", 2)):
        assert shapeSize(shape) == TensorData(shape).size
