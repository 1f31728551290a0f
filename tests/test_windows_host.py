"""x[key] of whole numbers and slices through the native module against the Python form, which arrays of a derived class take: the same
views, the same refusals. Views are arithmetic on shapes and steps: no device."""
import itertools

import numpy as np
import pytest

import cumo_amd as m


class DerivedSFloat(m.SFloat):
    pass


class DerivedBit(m.Bit):
    pass


PARTS = [0, 3, -1, -7, True, False, slice(None), slice(None, None, 2), slice(None, None, -1), slice(5, 1, -2), slice(-3, None), slice(2, 2), slice(9, 100),
         slice(None, None, 10 ** 30), slice(-10 ** 30, 10 ** 30, 3), np.int64(1), slice(np.int64(1), None), Ellipsis, 6, 7, 10 ** 30]


def view_of(cls, shape, key):
    a = cls(*shape, _buffer=m._native.Buffer(0), _offset=64)
    a = a._view(a.shape[::-1], a._strides[::-1], a._offset)   # the last dimension the slow one
    try:
        v = a[key]
    except (IndexError, TypeError, ValueError, OverflowError) as e:
        return type(e)
    return v.shape, v._strides, v._offset, type(v) is cls, v._buf is a._buf


@pytest.mark.parametrize("cls, derived", [(m.SFloat, DerivedSFloat), (m.Bit, DerivedBit)])
def test_windows_are_what_the_general_form_gives(cls, derived):
    keys = PARTS + [()] + [(k,) for k in PARTS] + list(itertools.product(PARTS, repeat=2)) + [(0, 1, 2), (slice(None), True, 0, 1), (slice(0, 1, 1), 1, slice(3))]
    for shape in ((7,), (4, 7), (2, 1, 7), (0, 7), ()):
        for key in keys:
            assert view_of(cls, shape, key) == view_of(derived, shape, key), (shape, key)


def test_a_step_of_zero_is_refused():
    for cls in (m.SFloat, DerivedSFloat):
        assert view_of(cls, (7,), slice(None, None, 0)) is ValueError


class Number:
    """A number of a slice whose __index__ is counted, and does something beside."""

    def __init__(self, value, beside=lambda: None):
        self.value, self.beside, self.asked = value, beside, 0

    def __index__(self):
        self.asked += 1
        self.beside()
        return self.value


@pytest.mark.parametrize("cls", [m.SFloat, DerivedSFloat, m.Bit, DerivedBit])
def test_a_slice_whose_numbers_set_the_array_anew(cls):
    """The view is of the array as it was when it was asked for; nothing is read from a shape that has gone."""
    def windows(beside):
        a = cls(5, 6, 7, 8, _buffer=m._native.Buffer(0), _offset=64)
        v = a[slice(Number(1, lambda: beside(a)), None), 2, slice(None, Number(-2)), ::3]
        return v.shape, v._strides, v._offset

    def nothing_left(a):
        a.shape, a._strides, a._offset = (), (), 0

    assert windows(nothing_left) == windows(lambda a: None)


@pytest.mark.parametrize("cls", [m.SFloat, DerivedSFloat])
def test_the_numbers_of_a_slice_are_asked_for_once(cls):
    a = cls(5, 6, 7, _buffer=m._native.Buffer(0))
    for rest in [(), (1,), (slice(2),), (Ellipsis,), (np.int64(1),), (0, 9), (10 ** 30,)]:
        n = Number(1)
        try:
            a[(slice(n, None),) + rest]
        except (IndexError, OverflowError):
            pass
        assert n.asked == 1, rest
