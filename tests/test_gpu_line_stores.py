"""Bilinear launches with planar outputs whose stores are moved on to line boundaries: which launches do (on the host), and on the GPU every
shift of a row and a channel plane, rows shorter than a step, partial last steps and workgroups, both numbers of lanes, streamed outputs, chains
compiled on first use and letterboxes.  Bit for bit the oracle's, and the strip form switched off gives the same."""
import numpy as np
import pytest

import fkl_cases as cases
import oracle_lib as ol
import workloads as wl


@pytest.mark.parametrize("w,h,planes,grain,lines", [
    (193, 105, 64, 4, 1), (193, 105, 64, 16, 0), (130, 60, 64, 8, 0), (75, 200, 64, 4, 1), (225, 225, 8, 4, 1), (99, 585, 8, 4, 0), (129, 530, 8, 4, 0), (179, 273, 8, 4, 1),
    (303, 307, 8, 4, 1), (300, 50, 64, 16, 1), (300, 50, 64, 32, 0), (467, 239, 8, 4, 0), (601, 600, 8, 4, 0), (639, 639, 64, 4, 1), (641, 641, 64, 4, 0),
    (224, 224, 64, 128, 0), (1, 1, 1, 4, 0)])
def test_which_launches_move_their_stores(w, h, planes, grain, lines):
    assert cases.cases().fklcase_lines_pay(w, h, planes, grain) == lines


def test_strips_of_a_plane_are_dealt_to_the_xcds_in_runs():
    """fkd::plane_band: every strip once, and XCD k, which has the workgroups of number k modulo 8, the k-th run of them in every plane."""
    band = cases.cases().fklcase_plane_band
    for gx in list(range(1, 75)) + [160, 251, 6001]:
        for z in (0, 1, 2, 7, 63):
            parts = [band(x, gx, z) for x in range(gx)]
            assert sorted(parts) == list(range(gx))
            xcd = {p: (z * gx + x) % 8 for x, p in enumerate(parts)}
            assert all(xcd[p] <= xcd[p + 1] for p in range(gx - 1)), (gx, z)


def image(w, h, seed):
    return np.random.RandomState(seed).randint(0, 256, (h, w, 3)).astype(np.uint8)


def rects_in(rng, n, w, h):
    r = np.zeros((n, 4), np.int32)
    for i in range(n):
        cw, ch = rng.randint(2, w + 1), rng.randint(1, h + 1)
        r[i] = (w - cw if i % 3 == 0 else rng.randint(0, w - cw + 1), h - ch if i % 2 == 0 else rng.randint(0, h - ch + 1), cw, ch)
    return r


# 32 lanes to a row (64 planes), 64 (8 planes), wide, streamed past the last-level cache
@pytest.mark.gpu
@pytest.mark.parametrize("batch,dst", [
    (64, (33, 350)), (64, (65, 190)), (64, (95, 121)), (64, (97, 118)), (64, (127, 91)), (64, (129, 89)), (64, (165, 77)), (64, (255, 71)),
    (8, (161, 301)), (8, (225, 226)), (8, (254, 233)), (8, (105, 901)), (64, (257, 33)), (8, (319, 250)), (64, (450, 33)), (64, (511, 34)), (64, (300, 41)),
    (64, (357, 310)), (64, (543, 203)), (64, (639, 171))])
@pytest.mark.parametrize("width", [201, 204])
def test_crops(device, batch, dst, width):
    import torch
    from fusedkernellibrary_amd import last_launch, lib
    assert cases.cases().fklcase_lines_pay(dst[0], dst[1], batch, 16 if dst[0] == 300 else 4) == 1
    rng = np.random.RandomState(dst[0])
    img, rects = image(width, 77, dst[1]), rects_in(np.random.RandomState(dst[1]), batch, width, 77)
    src = torch.from_numpy(img).to(device)
    n = batch * 3 * dst[1] * dst[0]
    # the output in the middle of a buffer, its first element anywhere between two line boundaries
    start = 64 + (dst[0] * 7 + width) % 32 if dst[0] != 300 else 64
    buf = torch.full((n + 128,), -7.0, dtype=torch.float32, device=device)
    out = buf[start:start + n].view(batch, 3, dst[1], dst[0])
    got = []
    for on in (1, 0):
        old = lib().fklhip_strip_form(on)
        try:
            buf.fill_(-7.0)
            cases.crop_resize_norm_split(src, rects, dst, wl.C3_MEAN, wl.C3_STD, out)
            torch.cuda.synchronize()
        finally:
            lib().fklhip_strip_form(old)
        ll = last_launch()
        assert ll["form"] == ("strip_lines" if on else "tiles")
        if on:
            # (narrow rows have 64 lanes where there would be few workgroups)
            lanes = 64 if dst[0] > 256 or (dst[1] + 7) // 8 * batch < 540 else 32
            assert ll["grid"] == [-(-dst[1] // (256 // lanes)), 1, batch] and ll["lds_bytes"] == (11 * 64 if lanes == 64 else 9 * 32) * 16 + 16
        got.append(buf.clone())
    assert torch.equal(got[0].view(torch.int32), got[1].view(torch.int32))
    assert (got[0][:start] == -7).all() and (got[0][start + n:] == -7).all()
    few = rng.choice(batch, 3, replace=False)
    for z in few:
        want = ol.oracle_crop_resize_norm_split(img, rects[z:z + 1], dst, wl.C3_MEAN, wl.C3_STD)
        assert got[0][start:start + n].view(batch, 3, dst[1], dst[0])[int(z)].cpu().numpy().tobytes() == want[0].tobytes(), z


@pytest.mark.gpu
@pytest.mark.parametrize("kind,cn,dtype", [(0, 2, np.uint8), (1, 4, np.uint8), (2, 3, np.uint16)])
@pytest.mark.parametrize("dst", [(255, 2300), (333, 2003), (511, 2001)])
def test_compiled_on_first_use(device, kind, cn, dtype, dst):
    import torch
    from fusedkernellibrary_amd import last_launch
    img = np.random.RandomState(60 + kind).randint(0, 1024 if dtype == np.uint16 else 256, (110, 203, cn)).astype(dtype)
    rect = (3, 2, 190, 100)
    src = torch.from_numpy(img.view(np.int16) if dtype == np.uint16 else img).to(device)
    out = torch.full((cn, dst[1], dst[0]), -7.0, dtype=torch.float32, device=device)
    cases.uncompiled_resize_split(kind, src, rect, dst, 0.5, out)
    torch.cuda.synchronize()
    ll = last_launch()
    assert ll["form"] == "strip_lines" and ll["block"] == [64, 4, 1] and ll["grid"] == [(dst[1] + 3) // 4, 1, 1]
    want = np.zeros((cn, dst[1], dst[0]), np.float32)
    ol.execute([ol.read_2d(img, cn, crop=rect, resize=dst, ar=ol.IGNORE_AR)], [ol.op(ol.MUL, (0.5, 0.5, 0.5, 0.5))],
               [ol.write(ol.TENSOR_SPLIT, want, cn, dst[0], dst[1], 1, cn)])
    assert out.cpu().numpy().tobytes() == want.tobytes()


@pytest.mark.gpu
@pytest.mark.parametrize("dst", [(101, 3001), (355, 670), (237, 801)])
def test_letterboxes(device, dst):
    import torch
    img = image(203, 99, 3)
    rects = np.array([[0, 0, 203, 99], [5, 3, 40, 90], [100, 90, 100, 9]], np.int32)
    bg, mul = np.float32([9, -8, 7]), np.float32([2, 0.5, 1.5])
    src = torch.from_numpy(img).to(device)
    out = torch.full((3, 3, dst[1], dst[0]), -7.0, dtype=torch.float32, device=device)
    from fusedkernellibrary_amd import last_launch, lib
    got = []
    for on in (1, 0):
        old = lib().fklhip_strip_form(on)
        try:
            out.fill_(-7.0)
            cases.uncompiled_letterbox_split_b3(src, rects, dst, bg, mul, out)
            torch.cuda.synchronize()
        finally:
            lib().fklhip_strip_form(old)
        assert last_launch()["form"] == ("strip_lines" if on else "tiles")
        got.append(out.cpu().numpy().tobytes())
    assert got[0] == got[1]
