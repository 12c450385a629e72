"""The tile form of the bilinear kernel in its three tile sizes (fkd::gather_form): which launch takes which, and for each the edges of waves and
tiles, sources at every alignment and rows up to the image's last, bit for bit against the oracle."""
import numpy as np
import pytest

import fkl_cases as cases
import oracle_lib as ol
from fusedkernellibrary_amd import last_launch

SUB, DIV = np.float32([103.5, 116.25, 123.0]), np.float32([57.0, 57.5, 58.25])


@pytest.mark.parametrize("w,h,planes,some,form", [
    (128, 8, 127, 920, 1), (128, 8, 128, 920, 2), (129, 8, 64, 920, 2), (128, 9, 63, 920, 1), (1, 1, 1, 920, 1), (128, 8, 919, 920, 2), (128, 8, 920, 920, 0),
    (1920, 1080, 1, 2560, 2), (2300, 1300, 1, 2560, 0), (1333, 800, 1, 2560, 2), (128, 64, 5, 920, 1), (640, 640, 64, 920, 0), (0, 5, 3, 920, 1)])
def test_form_by_number_of_tiles(w, h, planes, some, form):
    assert cases.cases().fklcase_gather_form(w, h, planes, some) == form


def image(w, h, seed):
    return np.random.RandomState(seed).randint(0, 256, (h, w, 3)).astype(np.uint8)


def rects_in(rng, n, w, h):
    r = np.zeros((n, 4), np.int32)
    for i in range(n):
        cw, ch = rng.randint(1, w + 1), rng.randint(1, h + 1)
        r[i] = (w - cw if i % 3 == 0 else rng.randint(0, w - cw + 1), h - ch if i % 2 == 0 else rng.randint(0, h - ch + 1), cw, ch)
    return r


# few tiles, some, many: the three forms
SIZES = ((1, 1), (2, 3), (63, 5), (64, 4), (65, 9), (127, 7), (128, 8), (129, 17), (192, 33), (257, 70), (300, 31), (385, 120), (290, 325))


@pytest.mark.gpu
@pytest.mark.parametrize("width", [91, 92])
def test_crops(device, width):
    import torch
    rng = np.random.RandomState(width)
    img = image(width, 77, 1)
    src = torch.from_numpy(img).to(device)
    for dst in SIZES:
        rects = rects_in(rng, 8, width, 77)
        out = torch.full((8, 3, dst[1], dst[0]), -1.0, dtype=torch.float32, device=device)
        cases.crop_resize_norm_split(src, rects, dst, SUB, DIV, out)
        torch.cuda.synchronize()
        assert out.cpu().numpy().tobytes() == ol.oracle_crop_resize_norm_split(img, rects, dst, SUB, DIV).tobytes(), dst


@pytest.mark.gpu
def test_default_planes(device):
    import torch
    rng = np.random.RandomState(3)
    img, default = image(120, 77, 2), np.float32([1, 2, 3])
    src = torch.from_numpy(img).to(device)
    for dst in SIZES:
        rects = rects_in(rng, 8, 120, 77)
        out = torch.full((8, 3, dst[1], dst[0]), -1.0, dtype=torch.float32, device=device)
        cases.crop_resize_default_norm_split(src, rects, dst, 3, default, SUB, DIV, out)
        torch.cuda.synchronize()
        assert out.cpu().numpy().tobytes() == ol.oracle_crop_resize_default_norm_split(img, rects, dst, 3, default, SUB, DIV).tobytes(), dst


@pytest.mark.gpu
def test_letterboxed_thumbnails(device):
    import torch
    rng = np.random.RandomState(5)
    img = image(203, 99, 3)
    src = torch.from_numpy(img).to(device)
    bg, mul, sub = np.float32([9, 8, 7]), np.float32([2, 2, 2]), np.float32([128, 100, 90])
    for dst in SIZES + ((300, 500),):
        rects = rects_in(rng, 5, 203, 99)
        out = torch.full((5, dst[1], dst[0], 3), 77, dtype=torch.uint8, device=device)
        cases.crop_resize_par_u8(src, rects, dst, bg, mul, sub, out)
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy(), ol.oracle_crop_resize_par_u8(img, rects, dst, bg, mul, sub)), dst


@pytest.mark.gpu
@pytest.mark.parametrize("size", [(64, 48), (46, 30)])
def test_nv12(device, size):
    """... the last two sizes are on both sides of the line for reads that convert every tap; with whole factors among them."""
    import torch
    w, h = size
    frame = np.random.RandomState(7).randint(0, 256, (h * 3 // 2, w)).astype(np.uint8)
    src = torch.from_numpy(frame).to(device)
    for dst in SIZES + ((32, 24), (23, 15), (2047, 1279), (2305, 1145)):
        out = torch.full((3, dst[1], dst[0]), -1.0, dtype=torch.float32, device=device)
        cases.nv12_rgb_resize_split(src, w, h, dst, np.float32(1 / 255), out)
        torch.cuda.synchronize()
        assert out.cpu().numpy().tobytes() == ol.oracle_nv12_rgb_resize_split(frame, w, h, dst, np.float32(1 / 255)).tobytes(), dst


@pytest.mark.gpu
def test_compiled_on_first_use(device):
    import torch
    img = np.random.RandomState(23).rand(40, 55, 4).astype(np.float32)
    src = torch.from_numpy(img).to(device)
    for dst in ((1, 1), (65, 5), (129, 9), (300, 500), (1025, 903), (1500, 800)):
        out = torch.full((dst[1], dst[0], 4), -1.0, dtype=torch.float32, device=device)
        cases.uncompiled_float4_resize(src, dst, out)
        torch.cuda.synchronize()
        assert last_launch()["kernel"] == "gather_jit"
        want = np.zeros((dst[1], dst[0], 4), np.float32)
        ol.execute([ol.read_2d(img, 4, resize=dst, ar=ol.IGNORE_AR)], [], [ol.write(ol.WRITE_2D, want, 4, dst[0], dst[1])])
        assert out.cpu().numpy().tobytes() == want.tobytes(), dst
