"""The grids of run-time compiled kernels (fkd::jit_geometry, on the host): whatever constants a module was compiled with, its workgroups cover every
row, column and element of the output, and no form launches a row of workgroups more than it needs."""
import ctypes as C
import itertools

import pytest

import fkl_cases as cases

GATHER, ROWS = 1, 0
STRIP, FLAT, SMALL = 1, 8, 4
SIZES = ((1, 1), (70, 33), (257, 9), (640, 480), (1500, 800), (1921, 1081), (75, 200), (4000, 3001))


def geometry(kind, w, h, planes, flags, v=4, rows=2, xi=2, yi=2, by=4, strip_width=256, bands=0, flat=1, whole=0):
    out = (C.c_uint * 6)()
    cases.cases().fklcase_jit_geometry((C.c_uint * 10)(kind, v, rows, xi, yi, by, strip_width, bands, flat, whole), w, h, planes, flags, out)
    return list(out)


def ceil(a, b):
    return -(-a // b)


@pytest.mark.parametrize("rows", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("flags", [0, SMALL])
def test_rows(rows, flags):
    for (w, h), planes in itertools.product(SIZES, (1, 5, 100)):
        which, gx, gy, waves, _, _ = geometry(ROWS, w, h, planes, flags, rows=rows)
        per_thread = {0: rows, 1: max(rows // 2, 1), 4: max(rows // 2, 1), 6: rows}[which]
        assert waves == 4 and gx == ceil(w, 256) and gy == ceil(h, 4 * per_thread), (w, h, planes)
        assert (which in (1, 6)) == bool(flags and w >= 4)


@pytest.mark.parametrize("rows", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("flags", [0, SMALL])
def test_planes_without_gaps(rows, flags):
    for (w, h), planes in itertools.product(SIZES, (1, 5, 100)):
        which, gx, gy, waves, _, _ = geometry(ROWS, w, h, planes, FLAT | flags, rows=rows)
        per_wave = {2: rows, 3: max(rows // 2, 1), 5: max(rows // 2, 1)}[which]
        assert waves == 4 and gy == 1 and gx == ceil(w * h, 64 * 4 * 4 * per_wave), (w, h, planes)


@pytest.mark.parametrize("h,blocks", [(511, 64), (4088, 511), (4096, 512), (8192, 1024), (8193, 1025), (16376, 2047), (16384, 2048)])
@pytest.mark.parametrize("flags", [0, FLAT])
def test_rows_per_thread_where_all_of_them_make_a_round(h, blocks, flags):
    """One column of workgroups of two rows: chains that keep their rows do so from two to four workgroups per compute unit, and no chain from 2048 on."""
    for whole in (0, 1):
        which, gx, gy, _, _, _ = geometry(ROWS, 256, h, 1, flags, whole=whole)
        all_rows = blocks >= 2048 or (whole and 512 <= blocks <= 1024)
        assert which == ((2 if all_rows else 5) if flags else (0 if all_rows else 4))
        assert gx * gy == (blocks if all_rows else ceil(h, 4))


@pytest.mark.parametrize("xi,yi", [(1, 1), (2, 2), (4, 1), (4, 3), (3, 2)])
def test_tiles(xi, yi):
    forms = set()
    for (w, h), planes in itertools.product(SIZES, (1, 8, 64)):
        which, gx, gy, waves, tx, ty = geometry(GATHER, w, h, planes, 0, xi=xi, yi=yi)
        form_xi, form_yi = {0: (xi, yi), 1: (1, 1), 2: (2, 1)}[which]
        assert (tx, ty) == (ceil(w, 64 * form_xi), ceil(h, waves * form_yi)) and gy == 1 and gx == ceil(tx * ty, 8) * 8, (w, h, planes)
        forms.add(which)
    assert forms == {0, 1, 2}


@pytest.mark.parametrize("xi,yi", [(1, 1), (2, 2), (4, 3)])
def test_strips_have_eight_rows_whatever_the_tiles(xi, yi):
    for h in (1, 7, 8, 9, 224, 640):
        assert geometry(GATHER, 224, h, 64, STRIP, xi=xi, yi=yi)[:3] == [0, ceil(h, 8), 1]
