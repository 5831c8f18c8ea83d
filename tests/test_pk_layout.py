"""The cached layout of the P(k) output vector: what the library refuses stays refused after an equal size was asked for."""
import ctypes

import pytest


def test_sizes_that_are_no_integers():
    from pylians_amd.Pk_library import pk_layout
    assert pk_layout(64) == pk_layout(64)
    with pytest.raises(ctypes.ArgumentError):
        pk_layout(64.0)
