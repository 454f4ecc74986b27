"""The plan of the kernels that stage two planes per wavefront, on the host: every geometry gets an answer, and every plan reaches every
pooled cell."""
import ctypes
import threading

import pytest

from convlogic_amd.hip import _lib


def _in_a_thread(work):
    """(the library's last error is the thread's: refused geometries leave none behind here)"""
    raised = []

    def run():
        try:
            work()
        except BaseException as e:
            raised.append(e)
    t = threading.Thread(target=run)
    t.start()
    t.join()
    if raised:
        raise raised[0]


def _check(lib, n, c_in, h, w, c_out, kh, kw, ph, pw, seen):
    g = _lib.ConvGeom(n, c_in, h, w, c_out, 1, 1, ph, pw, kh, kw)
    ho, wo = h + 2 * ph - kh + 1, w + 2 * pw - kw + 1
    fine = ho > 0 and wo > 0 and ho % 2 == 0 and wo % 2 == 0
    for dtype in (0, 1):
        for size in (lib.clg_convblock_forward_scratch_bytes, lib.clg_convblock_backward_scratch_bytes):
            assert (size(dtype, ctypes.byref(g)) >= 0) == fine
    assert (lib.clg_convblock_eval_packed_scratch_bytes(ctypes.byref(g)) >= 0) == fine
    plan = (ctypes.c_int64 * 6)()
    for dtype, weight_gradient in ((0, 0), (1, 0), (0, 1)):
        took = lib.clg_convblock_pair_plan(dtype, ctypes.byref(g), weight_gradient, plan)
        assert (took >= 0) == fine
        if took != 1:
            continue
        samples, groups, bands, rows, lds, parts = plan
        cells, pieces_in_rows = (ho // 2) * (wo // 2), w % (4 if dtype == 0 else 2) == 0
        assert 0 < lds <= 64 * 1024
        assert weight_gradient or groups * -(-c_out // 64) < 2**24    # (workgroups of 256 threads; at most 64 kernels each)
        if bands:                                                     # a lane per cell of a band, the bands cover the rows, none is empty
            assert weight_gradient == 0 and samples == 1 and groups == n * bands
            assert rows * (wo // 2) <= 64 and bands * rows >= ho // 2 > (bands - 1) * rows
        else:                                                         # more cells than lanes: only the kernels that walk a group
            assert samples * groups >= n > samples * (groups - 1)
            assert samples * cells <= 64 or weight_gradient or not pieces_in_rows
        if weight_gradient:                                           # terms a lane adds to one sum: no more than in the kernel of the padded copy
            blocks, total = -(-samples * cells // 64), n * cells
            other = -(-total // (256 * min(64, -(-total // (256 * (16 if total >= 65536 else 8))))))
            assert 1 <= parts <= 64 and (parts == 64 or -(-groups // (4 * parts)) * blocks <= max(other, blocks))
        seen.add((dtype, weight_gradient, bands > 0, samples * cells > 64))


@pytest.mark.timeout(120)
def test_plans_of_all_small_geometries():
    # (a row length that is no multiple of a 16-byte piece once left the search for a sample stride without an end: images of 8 x 7
    # with a 3 x 4 kernel)
    seen = set()

    def work():
        lib = _lib.load()
        for n in (1, 9, 100):
            for h in range(2, 35):
                for w in range(2, 35):
                    for kernel in ((3, 3, 1, 1), (3, 4, 1, 1), (4, 3, 1, 2), (5, 5, 2, 2), (2, 3, 0, 1)):
                        _check(lib, n, 5, h, w, 40, *kernel, seen)
    _in_a_thread(work)
    assert {(0, 0, True, True), (0, 0, False, False), (0, 0, False, True), (1, 0, True, True), (0, 1, False, True)} <= seen


def test_parts_of_a_weight_gradient_of_many_kernels():
    def work():
        lib = _lib.load()
        for n in (1, 16, 33, 90, 128, 300, 400, 1000, 4096, 20000):
            for side in (4, 6, 8, 12, 16, 20, 24, 32):
                for c_out in (3, 64, 600, 1024, 4096, 65535):
                    _check(lib, n, 16, side, side, c_out, 3, 3, 1, 1, set())
    _in_a_thread(work)


def test_plans_of_wide_images():
    # rows of 64 cells and more: with whole pieces in a row they were once taken for bands of no rows, and nothing was written
    seen = set()

    def work():
        lib = _lib.load()
        for n, c_in, c_out in ((1, 3, 8), (64, 32, 64), (2**23, 3, 8)):
            for h in (2, 3, 4, 5, 6, 8, 16):
                for w in (*range(60, 70), *range(120, 140), 160, 200, *range(250, 264), 384, 512, 520):
                    for kernel in ((3, 3, 1, 1), (5, 5, 2, 2), (2, 2, 0, 0), (3, 4, 1, 1)):
                        _check(lib, n, c_in, h, w, c_out, *kernel, seen)
    _in_a_thread(work)
    assert {(0, 0, True, True), (0, 0, False, True), (0, 1, False, True)} <= seen
