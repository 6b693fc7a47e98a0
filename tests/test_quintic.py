"""Closest points of cubic segments (diffvg_amd/csrc/dvg_quintic.h, built for the host from the
header the GPU kernels compile) against the oracle's restatement of the reference's searches."""
import ctypes
import os

import pytest

SO = os.path.join(os.path.dirname(os.path.abspath(__file__)), 'csrc', 'libquintic_check.so')


@pytest.mark.parametrize('mode, large', [(0, 0.0), (1, 0.9), (2, 0.9), (3, 0.0), (4, 0.0), (5, 0.0), (6, 0.0), (7, 0.0),
                                         (8, 0.0), (9, 0.3), (10, 0.0), (11, 0.9), (12, 0.3), (13, 0.1),
                                         (14, 0.9), (15, 0.9), (16, 0.0)])
def test_closest_points_are_the_reference_s(mode, large):
    """A search that finds other roots than the reference's moves the distance by pixels; one
    that stops at another iterate (both stop once the polynomial is below 1e-5) moved it by at
    most 1.8e-4 over 30 million cases, so 1e-3 tells them apart.  `large`: the share that must
    take the plain search for the mode to mean anything."""
    if not os.path.exists(SO):
        pytest.skip('tests/csrc not built (make -C tests/csrc)')
    L = ctypes.CDLL(SO)
    L.quintic_fuzz.argtypes = [ctypes.c_int, ctypes.c_int64, ctypes.c_uint64, ctypes.POINTER(ctypes.c_int64),
                               ctypes.POINTER(ctypes.c_float)]
    out = (ctypes.c_int64 * 4)()
    worst = ctypes.c_float()
    L.quintic_fuzz(mode, 300000, 40 + mode, out, ctypes.byref(worst))
    assert out[2] == 0, (out[2], worst.value)
    assert out[3] == 0
    assert out[1] >= large * out[0]
