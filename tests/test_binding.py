"""The ctypes binding: a pointer passed to a call keeps its array, also one that nothing else refers to."""
import weakref

import numpy as np
import pytest

import maplemoe as M
import pyoracle as O


@pytest.mark.parametrize("ptr", [M.ptr, O._p])
def test_pointer_holds_a_temporary(ptr):
    a = np.arange(16, dtype=np.float32)
    alive = weakref.ref(a)
    p = ptr(a)
    del a
    assert alive() is not None and p.value == alive().ctypes.data
    del p
    assert alive() is None
    assert ptr(None) is None
