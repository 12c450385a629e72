"""Warps whose lanes own one column of four output rows (scattered reads of the rows kernel): the edges of a wave's 64 columns and of a
block's 256x4 outputs, segments that begin where a line does, workgroups renumbered inside a two-dimensional grid, the split
between waves inside the source and others, batches, and coordinates at the very edge of the source.  Bit for bit the
oracle's, and no byte beside the output is written."""
import math

import numpy as np
import pytest

import fkl_cases as cases
import oracle_lib as ol
from test_gpu_any_alignment import Placed

pytestmark = pytest.mark.gpu

AFFINE = [[0.9 * math.cos(0.3), -0.9 * math.sin(0.3), 30.5], [0.9 * math.sin(0.3), 0.9 * math.cos(0.3), -17.25]]
PERSPECTIVE = [[1.1, 0.05, -3.0], [0.02, 0.9, 4.0], [0.0002, -0.0001, 1.0]]


def image(w, h, seed=3):
    return np.random.RandomState(seed).randint(0, 256, (h, w, 3)).astype(np.uint8)


def check(device, img, matrix, persp, dst, offset=0, pad=0):
    import torch
    out = Placed((dst[1], dst[0], 3), np.float32, offset, pad, device)
    cases.warp(torch.from_numpy(img).to(device), matrix, persp, dst, out.view())
    torch.cuda.synchronize()
    want = ol.oracle_warp(img, 3, matrix, dst, persp)
    assert out.read().tobytes() == want.tobytes(), (img.shape, dst, offset, pad)


@pytest.mark.parametrize("matrix,persp", [(AFFINE, False), (PERSPECTIVE, True)])
@pytest.mark.parametrize("height", [1, 2, 3, 4, 5, 9])
def test_edges_of_waves_and_blocks(device, matrix, persp, height):
    for n, width in enumerate((1, 2, 63, 64, 65, 127, 129, 255, 256, 257, 321, 513)):
        check(device, image(300, 200), matrix, persp, (width, height), 4 * (n % 4), (0, 4, 12)[n % 3])


@pytest.mark.parametrize("offset,pad", [(0, 0), (4, 0), (64, 0), (20, 4), (0, 84)])
def test_segments_from_line_boundaries(device, offset, pad):
    """26 MB of output with rows off the line boundaries: segments that begin left of a row, and one more at its right end."""
    dst = (1279, 1701)
    check(device, image(400, 300), AFFINE, False, dst, offset, pad)


@pytest.mark.parametrize("matrix,persp", [(AFFINE, False), (PERSPECTIVE, True)])
@pytest.mark.parametrize("dst", [(255, 1500), (257, 511), (257, 512), (771, 263), (1025, 205), (600, 999)])
def test_bands_inside_a_two_dimensional_grid(device, matrix, persp, dst):
    """Below, at and above the 256 blocks from which they are formed, with counts that leave every remainder of eight."""
    from fusedkernellibrary_amd import last_launch
    check(device, image(500, 400), matrix, persp, dst)
    assert last_launch()["grid"] == [(dst[0] + 255) // 256, (dst[1] + 3) // 4, 1]


@pytest.mark.parametrize("shape", [(1, 1), (1, 9), (2, 1), (2, 2), (3, 2), (700, 2), (2050, 2050)])
def test_waves_inside_and_at_the_edges(device, shape):
    """4 300 blocks (the form with a copy of the work for waves that are inside throughout) over sources of which nothing, a row or
    nearly everything counts as inside, and whose last column and row are met from both sides."""
    w, h = shape
    s = [[w / 2100.0, 0.0, 0.0], [0.0, h / 2100.0, 0.0]]
    check(device, image(w, h), s, False, (2100, 2100))


@pytest.mark.parametrize("matrix", [[[-1, -1, -0.0], [-1, -1, -0.0]], [[1, 0, float("nan")], [0, 1, 0]], [[1, 0, 0], [0, 1, float("inf")]],
                                    [[1, 0, -1e-30], [0, 1, 0]], [[1e30, 0, 0], [0, 1e30, 0]], [[1, 0, 1e-30], [0, 1, 1e-30]]])
def test_points_on_the_boundary(device, matrix):
    """Minus zero is inside; the smallest number below it, NaN and infinity are not."""
    check(device, image(67, 5), matrix, False, (67, 5))


def test_batch(device):
    import torch
    imgs = [image(131, 90, k) for k in range(3)]
    mats = [AFFINE, [[1, 0, 40], [0, 1, 0]], [[0.4, 0.1, 0], [-0.1, 0.4, 20]]]
    for dst in ((70, 6), (300, 1030), (1283, 709)):
        out = torch.full((3, dst[1], dst[0], 3), -1.0, dtype=torch.float32, device=device)
        cases.warp_batch([torch.from_numpy(i).to(device) for i in imgs], mats, dst, out)
        torch.cuda.synchronize()
        got = out.cpu().numpy()
        for k in range(3):
            assert got[k].tobytes() == ol.oracle_warp(imgs[k], 3, mats[k], dst, False).tobytes(), (dst, k)


@pytest.mark.parametrize("dst", [(65, 9), (1283, 1301)])
def test_single_floats(device, dst):
    import torch
    img = np.random.RandomState(4).rand(300, 400).astype(np.float32) * 10 - 5
    out = Placed((dst[1], dst[0]), np.float32, 8, 4, device)
    cases.warp(torch.from_numpy(img).to(device), AFFINE, False, dst, out.view())
    torch.cuda.synchronize()
    assert out.read().tobytes() == ol.oracle_warp(img, 1, AFFINE, dst, False).tobytes()
