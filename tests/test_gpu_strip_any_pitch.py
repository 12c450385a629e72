"""The strip form of the bilinear kernel on images whose rows do not share their alignment: bit for bit the oracle's result and the
tile form's, at every alignment of the image, with enlarging planes (columns clamped to the last one), letterboxes and crops that
end with the image.  (The bytes its tap windows touch: test_tap_windows.py.)"""
import numpy as np
import pytest

import fkl_cases as cases
import oracle_lib as ol
import workloads as wl
from test_gpu_any_alignment import Placed


def _view(img, offset, pad, device):
    import torch
    h, w = img.shape[:2]
    pitch = 3 * w + pad
    host = np.zeros(offset + pitch * h + 16, np.uint8)
    np.lib.stride_tricks.as_strided(host[offset:], (h, 3 * w), (pitch, 1))[:] = img.reshape(h, 3 * w)
    return torch.from_numpy(host).to(device)[offset:].as_strided((h, w, 3), (pitch, 3, 1), offset)


@pytest.mark.gpu
@pytest.mark.parametrize("batch,dst,form", [(64, (224, 224), "strip"), (8, (224, 264), "strip"), (64, (256, 61), "strip"), (8, (97, 130), "strip"),
                                            (64, (33, 190), "strip"), (8, (160, 32), "strip"), (8, (64, 40), "gather"), (8, (224, 61), "gather"),
                                            (64, (225, 61), "gather")])
@pytest.mark.parametrize("w,offset,pad", [(333, 0, 0), (1279, 1, 0), (334, 3, 1), (335, 2, 2), (253, 0, 7)])
def test_crops(device, batch, dst, form, w, offset, pad):
    import torch
    from fusedkernellibrary_amd import last_launch, lib
    rng = np.random.RandomState(w + batch + dst[0])
    h = 201
    img = rng.randint(0, 256, (h, w, 3)).astype(np.uint8)
    src = _view(img, offset, pad, device)
    rects = np.zeros((batch, 4), np.int32)
    for i in range(batch):
        cw, ch = rng.randint(2, w + 1), rng.randint(1, h + 1)
        rects[i] = (rng.randint(0, w - cw + 1), rng.randint(0, h - ch + 1), cw, ch)
    rects[0], rects[1], rects[2] = (0, 0, w, h), (w - 2, h - 2, 2, 2), (w - 40, h - 1, 40, 1)
    got = []
    for on in (1, 0):
        lib().fklhip_strip_form(on)
        try:
            out = torch.full((batch, 3, dst[1], dst[0]), -7.0, dtype=torch.float32, device=device)
            cases.crop_resize_norm_split(src, rects, dst, wl.C3_MEAN, wl.C3_STD, out)
            torch.cuda.synchronize()
            assert last_launch()["kernel"] == (form if on else "gather")
            got.append(out.cpu().numpy())
        finally:
            lib().fklhip_strip_form(1)
    want = ol.oracle_crop_resize_norm_split(img, rects, dst, wl.C3_MEAN, wl.C3_STD)
    assert got[0].tobytes() == want.tobytes() and got[1].tobytes() == want.tobytes()


@pytest.mark.gpu
@pytest.mark.parametrize("w,offset", [(321, 0), (322, 1), (323, 2)])
def test_letterboxes_compiled_on_first_use(device, w, offset):
    import torch
    from fusedkernellibrary_amd import last_launch
    rng = np.random.RandomState(w)
    img = rng.randint(0, 256, (200, w, 3)).astype(np.uint8)
    rects = np.array([[10, 20, 300, 60], [40, 0, 50, 200], [w - 120, 80, 120, 120]], np.int32)
    bg, mul = np.array([0.25, 128.5, 255.0], np.float32), np.array([0.5, 2.0, 1.0 / 255.0], np.float32)
    dst = (160, 300)
    out = torch.full((3, 3, dst[1], dst[0]), -7.0, dtype=torch.float32, device=device)
    cases.uncompiled_letterbox_split_b3(_view(img, offset, 0, device), rects, dst, bg, mul, out)
    torch.cuda.synchronize()
    assert last_launch()["kernel"] == "strip_jit"
    want = np.zeros((3, 3, dst[1], dst[0]), np.float32)
    reads = [ol.read_2d(img, 3, crop=rects[i], resize=dst, ar=ol.PRESERVE_AR, bg=tuple(bg) + (0.0,)) for i in range(3)]
    ol.execute(reads, [ol.op(ol.MUL, tuple(mul) + (0.0,))], [ol.write(ol.TENSOR_SPLIT, want, 3, dst[0], dst[1], 3, 3)])
    assert out.cpu().numpy().tobytes() == want.tobytes()


# Pixels whose tap pair is shifted into place inside its window (2 and 6 bytes) and pixels of whole dwords, whose pair is fetched
# from exactly where it begins: every address and pitch that leaves the samples aligned.
@pytest.mark.gpu
@pytest.mark.parametrize("kind,cn,dtype", [(0, 2, np.uint8), (1, 4, np.uint8), (2, 3, np.uint16)])
@pytest.mark.parametrize("w,dst,rect", [(201, (160, 256), (3, 1, 190, 90)), (202, (97, 430), (0, 0, 202, 110)),
                                        (203, (64, 640), (200, 108, 3, 2))])             # the last one enlarges the image's last pixels
def test_other_pixel_types(device, kind, cn, dtype, w, dst, rect):
    import torch
    from fusedkernellibrary_amd import last_launch, lib
    size, h = np.dtype(dtype).itemsize, 110
    img = np.random.RandomState(60 + kind).randint(0, 1024 if size == 2 else 256, (h, w, cn)).astype(dtype)
    want = np.zeros((cn, dst[1], dst[0]), np.float32)
    ol.execute([ol.read_2d(img, cn, crop=rect, resize=dst, ar=ol.IGNORE_AR)], [ol.op(ol.MUL, (0.5, 0.5, 0.5, 0.5))],
               [ol.write(ol.TENSOR_SPLIT, want, cn, dst[0], dst[1], 1, cn)])
    wrong = []
    for offset in range(0, 4, size):
        for pad in range(0, 4, size):
            src = Placed(img.shape, dtype, offset, pad, device, img)
            for on in (1, 0):
                old = lib().fklhip_strip_form(on)
                try:
                    out = torch.full((cn, dst[1], dst[0]), -7.0, dtype=torch.float32, device=device)
                    cases.uncompiled_resize_split(kind, src.view(), rect, dst, 0.5, out)
                    torch.cuda.synchronize()
                    assert last_launch()["kernel"] == ("strip_jit" if on else "gather_jit")
                finally:
                    lib().fklhip_strip_form(old)
                if out.cpu().numpy().tobytes() != want.tobytes():
                    wrong.append((offset, src.pitch, on))
    assert not wrong
