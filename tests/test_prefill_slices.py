"""The K slices of a prefill logits launch (dsa_prefill_slice_pages), on the host: the slice of least cost over every
length, within the 255-page block-table stage; few enough lengths tried that a small call does not wait for it."""
import ctypes
import os
import time

import pytest

import hcu_ops

STAGE = 255  # pages of a CTA's block-table slice


@pytest.fixture(scope="module")
def slice_pages():
    lib = ctypes.CDLL(os.path.join(os.path.dirname(hcu_ops.__file__), "libdsa_indexer.so"))
    f = lib.dsa_prefill_slice_pages
    f.argtypes = [ctypes.c_int, ctypes.c_int64, ctypes.c_int64, ctypes.c_int]
    return f


def cheapest(heads, groups, pages, cus):
    """The first slice length of least cost (sixths of a page); for 64 heads the longest slices from a group and 2048
    pages a CU on."""
    if heads == 64 and groups >= cus and groups * pages >= 2048 * cus:
        n = -(-pages // STAGE)
        return -(-pages // n)

    def cost(length):
        rounds = -(-groups * -(-pages // length) // cus)
        return rounds * (length + 1) * (8 if rounds == 1 else 6) + 3 * length

    return min(range(1, min(STAGE, pages) + 1), key=lambda length: (cost(length), length))


def test_slices_are_the_cheapest(slice_pages):
    for cus in (64, 256):
        for groups in (1, 2, 7, 33, 64, 113, 256, 511, 512, 626, 2048):
            for pages in (1, 2, 17, 64, 79, 128, 255, 256, 328, 501, 939, 1023, 1024, 1152, 2304):
                for heads in (32, 64):
                    got = slice_pages(heads, groups * 8, pages * 64, cus)
                    assert got == cheapest(heads, groups, pages, cus), (heads, groups, pages, cus)
                    assert 1 <= got <= STAGE


def test_few_rows_are_one_launch(slice_pages):
    """1, 2 and 4 rows share the pages evenly (0); three rows are a short 8-row group, not launches of two and one
    that read every key twice."""
    for heads in (32, 64):
        for width in (100, 30004, 65472):
            assert [slice_pages(heads, rows, width, 256) > 0 for rows in range(0, 10)] == [False] * 3 + [True, False] + [True] * 5
    assert slice_pages(32, 4, 65537, 256) > 0 and slice_pages(64, 4, 65537, 256) == 0


def test_rule_costs_little_host_time(slice_pages):
    def ns(rows, width):
        best = None
        for _ in range(15):
            t = time.perf_counter()
            for _ in range(500):
                slice_pages(64, rows, width, 256)
            t = (time.perf_counter() - t) / 500 * 1e9
            best = t if best is None else min(best, t)
        return best

    # 95 ns past the call itself; 1860 with every length tried
    assert ns(64, 60064) - ns(4, 60064) < 800
