"""Warps over a rectangle of an image: the rectangle's own first row and column, for every kind of pixel with paired taps, with an
operation fused into the read on either side of the crop, single and batched, ahead of time (affine uchar3) and compiled on first use, in
small launches and in those that are renumbered into bands.  Bit for bit the oracle's."""
import math

import numpy as np
import pytest

import fkl_cases as cases
import oracle_lib as ol

pytestmark = pytest.mark.gpu

W, H = 163, 120
RECTS = ((0, 0, W, H), (3, 0, 70, 60), (0, 1, 90, 50), (41, 20, 100, 77), (40, 21, 101, 60), (W - 50, H - 40, 50, 40), (W - 2, H - 1, 2, 1))
MUL = np.float32([0.5, 1.25, 3.0])
KINDS = {0: (np.uint8, 3), 1: (np.float32, 1), 2: (np.uint16, 3), 3: (np.uint8, 3), 4: (np.uint8, 3)}


def matrix(rect, dst, persp):
    """A turn by 0.3 about the middles that takes the rectangle to somewhat more than the output."""
    s, c, d = 1.1 * rect[2] / dst[0], math.cos(0.3), math.sin(0.3)
    sy = 1.1 * rect[3] / dst[1]
    m = [[s * c, -s * d, rect[2] / 2 - (s * c * dst[0] - s * d * dst[1]) / 2], [sy * d, sy * c, rect[3] / 2 - (sy * d * dst[0] + sy * c * dst[1]) / 2]]
    return m + [[0.05 / dst[0], -0.03 / dst[1], 1.0]] if persp else m


def image(kind):
    dtype, cn = KINDS[kind]
    rng = np.random.RandomState(kind)
    shape = (H, W, cn) if cn > 1 else (H, W)
    if dtype == np.float32:
        return (rng.rand(*shape) * 10 - 5).astype(dtype)
    return rng.randint(0, 1000 if dtype == np.uint16 else 256, shape).astype(dtype)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("persp", [False, True])
def test_rectangles(device, kind, persp):
    import torch
    img = image(kind)
    src = torch.from_numpy(img.view(np.int16) if img.dtype == np.uint16 else img).to(device)
    tap_ops = [ol.op(ol.MUL, MUL)] if kind >= 3 else None
    wrong = []
    # one block, several, and bands in a two-dimensional grid; then bands in a one-dimensional one
    for rect, dst in [(r, d) for r in RECTS for d in ((70, 50), (300, 64), (520, 523))] + [(RECTS[3], (2048, 2051))]:
        shape = (dst[1], dst[0], 3) if img.ndim == 3 else (dst[1], dst[0])
        out = torch.full(shape, -1.0, dtype=torch.float32, device=device)
        m = matrix(rect, dst, persp)
        cases.warp_crop(kind, src, rect, MUL, m, persp, dst, out)
        torch.cuda.synchronize()
        want = ol.oracle_warp(img, img.shape[2] if img.ndim == 3 else 1, m, dst, persp, crop=rect, tap_ops=tap_ops)
        if out.cpu().numpy().tobytes() != want.tobytes():
            wrong.append((rect, dst))
    assert not wrong


@pytest.mark.parametrize("dst", [(70, 50), (520, 523)])
def test_batch(device, dst):
    import torch
    img, rects = image(0), [RECTS[3], RECTS[5], RECTS[0]]
    m = matrix(RECTS[4], dst, False)
    out = torch.full((3, dst[1], dst[0], 3), -1.0, dtype=torch.float32, device=device)
    cases.warp_crops(torch.from_numpy(img).to(device), rects, m, dst, out)
    torch.cuda.synchronize()
    assert [r for got, r in zip(out.cpu().numpy(), rects) if got.tobytes() != ol.oracle_warp(img, 3, m, dst, False, crop=r).tobytes()] == []
