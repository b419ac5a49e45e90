"""The host rules of the direct sums (stkfmm_amd/csrc/p2p_direct_layout.hpp, p2p_internal.hpp), compiled for the CPU
by tests/cxx/direct_layout_host.cpp."""
import ctypes
import os

import numpy as np
import pytest

from tests.conftest import ROOT

LIB = os.path.join(ROOT, "tests", "cxx", "libdirect_layout_host.so")


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(LIB):
        pytest.skip("tests/cxx/libdirect_layout_host.so not built (make -C stkfmm_amd/csrc)")
    return ctypes.CDLL(LIB)


def view(first_double, stride, fstride=1):
    return (ctypes.c_ulonglong * 3)(2 ** 20 + 8 * first_double, stride, fstride)


def perm_rows(rows):
    """The permutation's presence and the rows it may reach."""
    return int(rows is not None), ctypes.c_longlong(-1 if rows is None else rows)


# the output's first double and rows [0, n_trg) x 3 against four inputs of 3 columns; a field of 6,000 rows of 3
# begins at double 0, other arrays lie at 100,000 and more
FAR = 200_000
OVERLAPS = [
    # out, rows a permutation may reach (None: no permutation, -1: not known), source values, overlap
    (0, None, FAR, False),
    (0, None, 0, True),
    (0, None, 2_999, True),          # the last value of row 999
    (0, None, 3_000, False),         # row 1,000
    (15_000, None, 12_000 - 1, False),
    (15_000, None, 12_000, False),   # rows [4,000, 5,000) before rows [5,000, 6,000)
    (15_000, None, 12_001, True),
    (0, -1, 15_000, True),           # rows 5,000 and on, through a permutation to the same rows
    (0, 6_000, 15_000, True),
    (0, 5_001, 15_000, True),
    (0, 5_000, 15_000, False),
    (0, 6_000, 0, True),
    (15_000, -1, 0, False),          # rows [0, 1,000): all in front of the output's first row
    (15_000, -1, 12_001, True),
    (0, 6_000, FAR, False),
    (0, -1, FAR, True),
    (FAR + 50_000, -1, FAR, False),
]


@pytest.mark.parametrize("out,rows,sv,expected", OVERLAPS)
@pytest.mark.parametrize("which", range(4))
def test_output_over_an_input_is_seen(lib, out, rows, sv, expected, which):
    """Each input in turn (source coordinates, first and second source values, target coordinates) where the output
    may be; the others in front of everything."""
    n = 1000
    arrays = [view(-100_000 + 4_000 * k, 3) for k in range(4)]
    arrays[which] = view(sv, 3)
    got = lib.direct_overlaps_host(*arrays, view(out, 3), *perm_rows(rows), n, n, 6, 3, 3)
    assert bool(got) == expected


def test_overlap_of_strided_views(lib):
    """Columns of one tensor of seven: the extents meet, whatever lies between them."""
    t = [view(100 * 7 * k + c, 7) for k, c in ((0, 0), (0, 3), (0, 6))]
    far = view(FAR, 3)
    assert lib.direct_overlaps_host(t[0], far, far, far, t[1], *perm_rows(None), 100, 100, 3, 3, 3)
    assert not lib.direct_overlaps_host(far, far, far, view(700, 7), t[1], *perm_rows(None), 100, 100, 3, 3, 3)
    # component-major: component 2 of 50 rows ends at double 149
    assert lib.direct_overlaps_host(view(0, 1, 50), far, far, far, view(149, 3), *perm_rows(None), 50, 50, 3, 3, 3)
    assert not lib.direct_overlaps_host(view(0, 1, 50), far, far, far, view(150, 3), *perm_rows(None), 50, 50, 3, 3, 3)


PARTIAL = 2 ** 21  # doubles of the partial-sum array


def layout(lib, prec, T, kt, n_src, n_trg, run=16, n_cu=256):
    out = (ctypes.c_int * 8)()
    lib.direct_layout_host(prec, T, kt, run, n_src, n_trg, n_cu, out)
    return dict(zip(("units", "chunks", "chunk_tiles", "waves", "unit", "ls", "tail_begin", "tail_ls"), out))


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("kt", [1, 3, 4, 6, 7, 10, 16])
def test_cut_covers_the_sum(lib, prec, kt):
    """Every target has a unit, every source tile a chunk, every chunk a tile; the chunks' sums fit their array."""
    rng = np.random.default_rng(10 * kt + prec)
    sizes = (10 ** rng.uniform(0, 6, (300, 2))).astype(int).tolist()
    for n_src, n_trg in sizes + [[1, 1], [64, 128], [65, 129], [16_000, 100_000], [4_000, 1_000_000]]:
        for T in (1, 2):
            c = layout(lib, prec, T, kt, n_src, n_trg)
            tiles = (n_src + 63) // 64
            assert c["chunks"] == 1 or c["chunks"] * n_trg * kt <= PARTIAL
            assert (c["chunks"] - 1) * c["chunk_tiles"] < tiles <= c["chunks"] * c["chunk_tiles"]
            whole = c["units"] - (1 if c["tail_ls"] else 0)
            assert (whole - 1) * c["unit"] < max(c["tail_begin"], 1) and whole * c["unit"] >= c["tail_begin"]
            assert c["tail_begin"] == n_trg or (prec and n_trg - c["tail_begin"] < 64 * T and c["tail_ls"])
            assert c["unit"] == 64 * T >> c["ls"] and 1 <= c["waves"] <= 8


# bounded by 131,072 targets' worth of chunks whatever the outputs: 6.05, 6.1, 6.1 and 3.7 workgroups a CU, whose
# last, partly filled round is as long as each of the others
@pytest.mark.parametrize("n_src,n_trg", [(16_000, 33_000), (16_000, 50_000), (16_000, 100_000), (120_000, 120_000)])
def test_targets_a_little_over_a_round(lib, n_src, n_trg):
    """Light kernels' sums whose units would be a little more than whole rounds of workgroups come in so many chunks
    that the last round is an eighth or less of the whole."""
    for prec in (0, 1):
        c = layout(lib, prec, 2, 4, n_src, n_trg)
        rounds = c["units"] * c["chunks"] / 256
        assert rounds >= 8, rounds


@pytest.mark.parametrize("n_src,n_trg,items", [(16_000, 500_000, True), (16_000, 268_435, False), (16_000, 268_436, True),
                                               (8_192, 524_287, False), (8_192, 524_288, True), (8_191, 600_000, False),
                                               (500_000, 16_000, False), (1_500, 3_000_000, False),
                                               (2 ** 30, 2 ** 30 - 1, False)])
def test_sums_that_go_to_the_items(lib, n_src, n_trg, items):
    got = lib.direct_items_pay_host(ctypes.c_longlong(n_src), ctypes.c_longlong(n_trg))
    assert bool(got) == items


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("T,kt,waves", [(1, 10, 0), (1, 16, 0), (2, 3, 0), (2, 6, 0), (1, 6, 8), (2, 3, 8)])
@pytest.mark.parametrize("n_trg", [2 ** 29, 2 ** 30 - 129, 2 ** 30 - 128, 2 ** 30 - 127, 2 ** 30 - 64])
def test_launches_stay_below_2_32_threads(lib, prec, T, kt, waves, n_trg):
    """The largest sums, and (eight waves a workgroup) the wall images' slabs of 2^29 targets."""
    out = (ctypes.c_longlong * 2)()
    assert lib.direct_sizes_host(2 ** 30, n_trg) and not lib.direct_sizes_host(1, 2 ** 30 - 63)
    for n_src in (1, 64, 300, 1_000, 20_000, 10 ** 6):
        lib.direct_threads_host(prec, T, kt, waves, n_src, n_trg, out)
        assert 0 < out[0] < 2 ** 32 and 0 < out[1] < 2 ** 32, (n_src, out[0], out[1])
