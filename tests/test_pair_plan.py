"""The plan of the kernels that stage two planes per wavefront, on the host: every geometry gets an answer."""
import ctypes

import pytest
import torch

from convlogic_amd.hip import _lib, convlogic_hip


@pytest.mark.timeout(60)
def test_scratch_sizes_of_all_small_geometries_come_back():
    # (a row length that is no multiple of a 16-byte piece once left the search for a sample stride without an end: images of 8 x 7
    # with a 3 x 4 kernel)
    lib = _lib.load()
    for n in (1, 9, 100):
        for h in range(2, 35):
            for w in range(2, 35):
                for kh, kw, ph, pw in ((3, 3, 1, 1), (3, 4, 1, 1), (4, 3, 1, 2), (5, 5, 2, 2), (2, 3, 0, 1)):
                    g = convlogic_hip._geom(torch.empty((n, 5, h, w), device="meta"), 40, 1, 1, ph, pw, kh, kw)
                    for dtype in (0, 1):
                        lib.clg_convblock_forward_scratch_bytes(dtype, ctypes.byref(g))
                        lib.clg_convblock_backward_scratch_bytes(dtype, ctypes.byref(g))
                    lib.clg_convblock_eval_packed_scratch_bytes(ctypes.byref(g))
