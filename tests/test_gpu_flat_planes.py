"""Launches that take a plane as one row, because the rows of what is read and of what is written follow each other without gaps: which
launches do (on the host), and on the GPU every remainder of a run, a wave and a workgroup, bases at any address, planes apart from each
other, small and large outputs, in place.  Results bit for bit, and no byte beside them is written."""
import numpy as np
import pytest

import fkl_cases as cases
import oracle_lib as ol
from fusedkernellibrary_amd import last_launch
from test_gpu_any_alignment import FILL, Placed

FLAT, SMALL = 8, 4
A = 0x7F0000000000


@pytest.mark.parametrize("w,h,planes,gap_in,gap_out,flat", [
    (40, 30, 2, 0, 0, True), (41, 31, 1, 0, 0, True), (40, 30, 2, 1, 0, False), (40, 30, 2, 0, 1, False), (40, 30, 1, 8, 8, False),
    (1, 4, 1, 0, 0, True), (4, 1, 3, 0, 0, True), (3, 1, 1, 0, 0, False), (1, 3, 1, 0, 0, False), (30000, 60000, 1, 0, 0, True),
    (46341, 46341, 1, 0, 0, False)])
def test_which_launches_are_flat(w, h, planes, gap_in, gap_out, flat):
    row = 3 * w
    flags = cases.copy_flags(A, (row + gap_in, (row + gap_in) * h % 2**31), A, (row + gap_out, (row + gap_out) * h % 2**31), w, h, planes)
    assert bool(flags & FLAT) == flat


@pytest.mark.parametrize("address,plane_gap,planes,h,bound", [
    (A, 0, 1, 5000, 0), (A + 1, 0, 1, 5000, 127), (A + 128, 1, 2, 5000, 127), (A + 128, 1, 1, 5000, 0), (A + 1, 0, 1, 100, 0)])
def test_where_segments_of_flat_launches_begin(address, plane_gap, planes, h, bound):
    """1024 uchar3 per row: at line boundaries where the output has more than 4 MiB and does not begin on one, and then there is
    no kernel for small outputs."""
    flags = cases.copy_flags(A, (3072, 3072 * h), address, (3072, 3072 * h + plane_gap), 1024, h, planes)
    assert flags >> 8 == bound and bool(flags & SMALL) == (h == 100) and flags & FLAT


SHAPES = ((1, 4), (5, 1), (1, 5), (3, 85), (1, 256), (257, 1), (7, 73), (1, 1023), (341, 3), (1025, 1), (5, 205), (2047, 1), (683, 3), (4097, 1),
          (11, 745), (8191, 1), (3, 4097))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", range(len(cases.TENSOR_KINDS)))
@pytest.mark.parametrize("in_place", [False, True])
def test_tensors_of_any_element(device, kind, in_place):
    import torch
    base, cn = cases.TENSOR_KINDS[kind]
    size = np.dtype(base).itemsize
    elem, planes = size * cn, 3
    # ... and one whose planes are 5 MB apart, not on line boundaries: segments that begin left of a plane
    for n, (w, h) in enumerate(SHAPES + ((1021, (5 << 20) // (1021 * elem * planes) + 1),)):
        row = w * elem
        data = np.random.RandomState(n).randint(0, 256, (planes, h * row)).astype(np.uint8)

        def place(offset, gap, fill):
            host = np.full(256 + offset + (h * row + gap) * planes + 256, FILL, np.uint8)
            at = np.lib.stride_tricks.as_strided(host[256 + offset:], (planes, h * row), (h * row + gap, 1))
            if fill:
                at[:] = data
            return host, at, (row, h * row + gap), 256 + offset

        out_host, out_at, out_pitches, out_start = place(size * (n % 5), size * (n % 4), in_place)
        out = torch.from_numpy(out_host).to(device)
        if in_place:
            cases.copy_tensor(kind, out[out_start:], out_pitches, out[out_start:], out_pitches, w, h, planes)
        else:
            src_host, _, src_pitches, src_start = place(size * (n % 3), size * (n % 2), True)
            cases.copy_tensor(kind, torch.from_numpy(src_host).to(device)[src_start:], src_pitches, out[out_start:], out_pitches, w, h, planes)
        torch.cuda.synchronize()
        assert last_launch()["form"] == ("flat" if w * h >= 4 else "rows")
        out_at[:] = data
        assert np.array_equal(out.cpu().numpy(), out_host), (w, h)


@pytest.mark.gpu
@pytest.mark.parametrize("offset", [0, 1, 2, 3])
def test_batches_of_images(device, offset):
    import torch
    rng = np.random.RandomState(offset)
    mul, add = rng.uniform(0.5, 2.0, (4, 3)).astype(np.float32), rng.uniform(-64, 64, (4, 3)).astype(np.float32)
    for w, h in SHAPES + ((1279, 719), (1283, 300)):
        imgs = [rng.randint(0, 256, (h, w, 3)).astype(np.uint8) for _ in range(4)]
        want = ol.oracle_batch_muladd_sat(imgs, mul, add)
        srcs = [Placed((h, w, 3), np.uint8, (offset + k) % 4, 0, device, a) for k, a in enumerate(imgs)]
        outs = [Placed((h, w, 3), np.uint8, (offset + 3 * k) % 128, 0, device) for k in range(4)]
        cases.batch_muladd_sat([s.view() for s in srcs], mul, add, [o.view() for o in outs])
        cases.batch_muladd_sat([s.view() for s in srcs], mul, add, [s.view() for s in srcs])      # in place
        torch.cuda.synchronize()
        assert last_launch()["form"] == "flat"
        for a, b, c in zip(srcs, outs, want):
            assert np.array_equal(b.read(), c) and np.array_equal(a.read(), c), (w, h, offset)


@pytest.mark.gpu
@pytest.mark.parametrize("n_ops", [1, 3, 100])
def test_float_chains(device, n_ops):
    import torch
    for n, (w, h) in enumerate(SHAPES + ((1283, 900), (2049, 2051))):
        img = np.random.RandomState(n).uniform(-1, 1, (h, w)).astype(np.float32)
        src, out = Placed((h, w), np.float32, 4 * (n % 4), 0, device, img), Placed((h, w), np.float32, 4 * (n % 3), 0, device)
        cases.add_mul_chain(src.view(), n_ops, 0.5, 1.0001, out.view())
        torch.cuda.synchronize()
        assert last_launch()["form"] == "flat"
        assert out.read().tobytes() == ol.oracle_add_mul_chain(img, n_ops, np.float32(0.5), np.float32(1.0001)).tobytes(), (w, h)


@pytest.mark.gpu
@pytest.mark.parametrize("pf,cr,cp,dtype", [(ol.PF_UYVY, 1, 1, np.uint8), (ol.PF_Y210, 0, 1, np.int16)])
def test_packed_video(device, pf, cr, cp, dtype):
    """Runs of packed 4:2:2 begin at even pixels whatever the output's address."""
    import torch
    for n, (w, h) in enumerate(((2, 2), (2, 3), (6, 43), (130, 2), (514, 1), (1026, 5), (1282, 301), (2, 4097))):
        frame = np.random.RandomState(n).randint(0, 256 if dtype == np.uint8 else 1024, (h, 2 * w)).astype(dtype)
        src = torch.from_numpy(frame).to(device)
        out = Placed((h, w, 3), np.float32, 4 * (n % 5), 0, device)
        cases.yuv_to_rgb(pf, cr, cp, src, w, h, out.view())
        torch.cuda.synchronize()
        assert last_launch()["form"] == "flat"
        assert out.read().tobytes() == ol.oracle_yuv_to_rgb(pf, cr, cp, frame.view(np.uint8 if dtype == np.uint8 else np.uint16), w, h).tobytes(), (w, h)


@pytest.mark.gpu
def test_planar_output(device):
    import torch
    for w, h in SHAPES + ((1279, 719),):
        img = np.random.RandomState(w).randint(0, 256, (h, w, 3)).astype(np.uint8)
        out = torch.full((3, h, w), -1.0, dtype=torch.float32, device=device)
        cases.u8x3_to_planes(torch.from_numpy(img).to(device), out)
        torch.cuda.synchronize()
        assert last_launch()["form"] == "flat"
        assert np.array_equal(out.cpu().numpy(), img.transpose(2, 0, 1).astype(np.float32)), (w, h)
