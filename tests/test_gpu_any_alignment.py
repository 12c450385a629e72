"""Rows of the pointwise chains at every byte alignment and every remainder of their width: images whose first byte, pitch and
width are anything, where a lane's run is one wide access at any address and the lane at a row's end works on the row's last run.
Results are the oracle's bit for bit and nothing beside the image is touched."""
import numpy as np
import pytest

import fkl_cases as cases
import oracle_lib as ol

pytestmark = pytest.mark.gpu

FILL = 0xA5


class Placed:
    """A (h, w, c) image in the middle of a device buffer of FILL bytes, `offset` bytes past an aligned address, rows `pitch`
    bytes apart."""
    def __init__(self, shape, dtype, offset, pad_bytes, device, data=None):
        import torch
        h, row = shape[0], int(np.prod(shape[1:])) * np.dtype(dtype).itemsize
        self.shape, self.dtype, self.row, self.pitch, self.start = shape, np.dtype(dtype), row, row + pad_bytes, 256 + offset
        host = np.full(self.start + self.pitch * h + 256, FILL, np.uint8)
        if data is not None:
            self._rows(host)[:] = np.ascontiguousarray(data).view(np.uint8).reshape(h, row)
        self.buf = torch.from_numpy(host).to(device)

    def _rows(self, host):
        return np.lib.stride_tricks.as_strided(host[self.start:], (self.shape[0], self.row), (self.pitch, 1))

    def view(self):
        """The image as the case drivers take it: a byte-strided tensor of its first row's address."""
        import torch
        size = self.dtype.itemsize
        kind = {1: torch.uint8, 2: torch.int16, 4: torch.float32}[size]
        assert self.start % size == 0 and self.pitch % size == 0
        inner = [int(np.prod(self.shape[i + 1:])) for i in range(1, len(self.shape))]
        return self.buf[self.start % size:self.buf.numel() // size * size].view(kind).as_strided(self.shape, [self.pitch // size] + inner, self.start // size)

    def read(self):
        host = self.buf.cpu().numpy()
        rows = self._rows(host)
        got = np.array(rows).view(self.dtype).reshape(self.shape)
        rows[:] = FILL
        assert (host == FILL).all(), "a byte beside the image was written"
        return got


WIDTHS = (1, 2, 3, 4, 5, 7, 9, 63, 255, 256, 257, 258, 259, 260, 511, 513, 1022, 1023)


@pytest.mark.parametrize("offset", [0, 1, 2, 3])
def test_uchar3_images(device, offset):
    import torch
    rng = np.random.RandomState(7 + offset)
    mul, add = rng.uniform(0.5, 2.0, (4, 3)).astype(np.float32), rng.uniform(-64, 64, (4, 3)).astype(np.float32)
    for n, w in enumerate(WIDTHS):
        h, pad = (1, 2, 9)[n % 3], (0, 1, 2, 5)[(n + offset) % 4]
        imgs = [rng.randint(0, 256, (h, w, 3)).astype(np.uint8) for _ in range(4)]
        want = ol.oracle_batch_muladd_sat(imgs, mul, add)
        srcs = [Placed((h, w, 3), np.uint8, offset, pad, device, a) for a in imgs]
        outs = [Placed((h, w, 3), np.uint8, (offset + 1) % 4, pad, device) for _ in imgs]
        cases.batch_muladd_sat([s.view() for s in srcs], mul, add, [o.view() for o in outs])
        cases.batch_muladd_sat([s.view() for s in srcs], mul, add, [s.view() for s in srcs])      # in place
        torch.cuda.synchronize()
        for a, b, c in zip(srcs, outs, want):
            assert np.array_equal(b.read(), c) and np.array_equal(a.read(), c), (w, h, pad, offset)


@pytest.mark.parametrize("n_ops", [1, 3, 100])
def test_float_chains(device, n_ops):
    import torch
    rng = np.random.RandomState(n_ops)
    for n, w in enumerate(WIDTHS):
        h, pad = (1, 3, 9)[n % 3], 4 * (n % 3)
        img = rng.uniform(-1, 1, (h, w)).astype(np.float32)
        src, out = Placed((h, w), np.float32, 4 * (n % 4), pad, device, img), Placed((h, w), np.float32, 4, pad, device)
        cases.add_mul_chain(src.view(), n_ops, 0.5, 1.0001, out.view())
        torch.cuda.synchronize()
        want = ol.oracle_add_mul_chain(img, n_ops, np.float32(0.5), np.float32(1.0001))
        assert out.read().tobytes() == want.tobytes(), (w, h, pad)


def test_streamed_launches(device):
    """More than 2^26 elements: the loads of every kind of wave carry the non-temporal hint."""
    import torch
    rng = np.random.RandomState(5)
    w, h = 1021, 661                                     # 100 * 1021 * 661 = 67 488 100
    img = [rng.randint(0, 256, (h, w, 3)).astype(np.uint8) for _ in range(2)]
    dev = [torch.from_numpy(a).to(device) for a in img]
    outs = torch.zeros((100, h, w, 3), dtype=torch.uint8, device=device)
    mul, add = rng.uniform(0.5, 2.0, (100, 3)).astype(np.float32), rng.uniform(-64, 64, (100, 3)).astype(np.float32)
    cases.batch_muladd_sat([dev[i % 2] for i in range(100)], mul, add, [outs[i] for i in range(100)])
    torch.cuda.synchronize()
    for i in (0, 1, 50, 99):
        want = ol.oracle_batch_muladd_sat([img[i % 2]], mul[i:i + 1], add[i:i + 1])[0]
        assert np.array_equal(outs[i].cpu().numpy(), want), i


@pytest.mark.parametrize("pf,cr,cp", [(ol.PF_NV12, 0, 1), (ol.PF_NV21, 0, 0), (ol.PF_P010, 0, 2), (ol.PF_P210, 1, 1), (ol.PF_Y210, 0, 1),
                                      (ol.PF_UYVY, 1, 1)])
def test_video_frames_to_rgb(device, pf, cr, cp):
    """Even widths (packed and semi-planar formats have no others), on both sides of a run, a wave and two waves."""
    import torch
    dt = np.uint16 if ol.PF_WIDE[pf] else np.uint8
    rng = np.random.RandomState(70 + pf)
    for n, w in enumerate((2, 4, 6, 10, 254, 256, 258, 260, 510, 514, 1022)):
        h, size = (2, 6, 12)[n % 3], np.dtype(dt).itemsize
        rows, cols = ol.frame_shape(pf, w, h)
        buf = rng.randint(0, 1024 if ol.PF_WIDE[pf] else 256, (rows, cols)).astype(dt)
        frame = Placed((rows, cols), dt, size * (n % 4), size * (n % 3), device, buf)
        out = Placed((h, w, 3), np.float32, 4 * (n % 4), 4 * (n % 2), device)
        cases.yuv_to_rgb(pf, cr, cp, frame.view(), w, h, out.view())
        torch.cuda.synchronize()
        assert out.read().tobytes() == ol.oracle_yuv_to_rgb(pf, cr, cp, buf, w, h).tobytes(), (w, h)


@pytest.mark.parametrize("w", [1, 255, 257, 511, 1023])
def test_warps(device, w):
    import torch
    rng = np.random.RandomState(w)
    img = rng.randint(0, 256, (61, 83, 3)).astype(np.uint8)
    m = np.array([[0.9, -0.2, 4.5], [0.15, 1.1, -3.25]], np.float32)
    for h in (1, 7):
        out = Placed((h, w, 3), np.float32, 4, 4, device)
        cases.warp(torch.from_numpy(img).to(device), m, False, (w, h), out.view())
        torch.cuda.synchronize()
        assert out.read().tobytes() == ol.oracle_warp(img, 3, m, (w, h), False).tobytes(), h


@pytest.mark.parametrize("pf,cr,cp", [(ol.PF_NV12, 0, 1), (ol.PF_NV21, 1, 0), (ol.PF_P010, 0, 2), (ol.PF_P210, 1, 1), (ol.PF_Y210, 0, 0),
                                      (ol.PF_UYVY, 1, 2)])
def test_rgb_to_video_frames(device, pf, cr, cp):
    """Both parities of both extents: the last chroma block of an odd one belongs to a single column or row.  Launches of
    2 048 workgroups and more give a thread two rows."""
    import torch
    dt = np.uint16 if ol.PF_WIDE[pf] else np.uint8
    size = np.dtype(dt).itemsize
    rng = np.random.RandomState(90 + pf)
    sizes = [(w, (1, 2, 5, 12)[n % 4]) for n, w in enumerate((1, 2, 3, 4, 5, 6, 7, 9, 254, 255, 256, 257, 258, 259, 260, 510, 513))]
    for n, (w, h) in enumerate(sizes + [(1021, 4100), (1026, 4097)]):
        rgb = rng.randint(0, 1024 if ol.PF_WIDE[pf] else 256, (h, w, 3)).astype(dt)
        rows, cols = ol.frame_shape(pf, w + (w & 1), h + (h & 1))
        if pf in (ol.PF_NV12, ol.PF_NV21, ol.PF_P010, ol.PF_P210):
            rows = h + (h + 1) // 2 if pf != ol.PF_P210 else 2 * h     # chroma rows start right after `height` luma rows
        start = np.full((rows, cols), 9, dt)
        frame = Placed((rows, cols), dt, size * (n % 4), size * (n % 3), device, start)
        src = Placed((h, w, 3), dt, size * ((n + 1) % 4), size * (n % 2), device, rgb)
        cases.rgb_to_yuv(pf, cr, cp, src.view(), frame.view())
        torch.cuda.synchronize()
        assert np.array_equal(frame.read(), ol.oracle_rgb_to_yuv(pf, cr, cp, rgb, start)), (w, h)


# Outputs of 6 MB and more (16 MB for uchar3, 24 MB for float3) with rows of 512 elements and more, whose waves' segments begin at line boundaries: whole lines, half
# lines and rows that all start on a boundary.
@pytest.mark.parametrize("w,h,pad", [(1921, 700, 1), (2051, 700, 0), (1924, 900, 2), (644, 2100, 2), (1024, 1400, 0)])
def test_line_aligned_segments_uchar3(device, w, h, pad):
    import torch
    rng = np.random.RandomState(w)
    mul, add = rng.uniform(0.5, 2.0, (4, 3)).astype(np.float32), rng.uniform(-64, 64, (4, 3)).astype(np.float32)
    imgs = [rng.randint(0, 256, (h, w, 3)).astype(np.uint8) for _ in range(4)]
    want = ol.oracle_batch_muladd_sat(imgs, mul, add)
    srcs = [Placed((h, w, 3), np.uint8, 3, pad, device, a) for a in imgs]
    outs = [Placed((h, w, 3), np.uint8, 0 if w == 1024 else i, 0 if w == 1024 else pad, device) for i in range(4)]
    cases.batch_muladd_sat([s.view() for s in srcs], mul, add, [o.view() for o in outs])
    cases.batch_muladd_sat([s.view() for s in srcs], mul, add, [s.view() for s in srcs])      # in place
    torch.cuda.synchronize()
    for a, b, c in zip(srcs, outs, want):
        assert np.array_equal(b.read(), c) and np.array_equal(a.read(), c)


@pytest.mark.parametrize("w,h,offset", [(1921, 1080, 4), (2049, 790, 0), (1536, 1000, 12), (1536, 1000, 0)])
@pytest.mark.parametrize("n_ops", [1, 100])
def test_line_aligned_segments_floats(device, n_ops, w, h, offset):
    import torch
    img = np.random.RandomState(w).uniform(-1, 1, (h, w)).astype(np.float32)
    src, out = Placed((h, w), np.float32, 0, 0, device, img), Placed((h, w), np.float32, offset, 0, device)
    cases.add_mul_chain(src.view(), n_ops, 0.5, 1.0001, out.view())
    torch.cuda.synchronize()
    assert out.read().tobytes() == ol.oracle_add_mul_chain(img, n_ops, np.float32(0.5), np.float32(1.0001)).tobytes()


@pytest.mark.parametrize("pf,cr,cp", [(ol.PF_NV12, 0, 1), (ol.PF_P010, 0, 2), (ol.PF_UYVY, 1, 1)])
@pytest.mark.parametrize("w,h,offset", [(966, 2080, 4), (2050, 1000, 8), (770, 2600, 0), (1280, 1600, 0)])
def test_line_aligned_segments_video_to_rgb(device, pf, cr, cp, w, h, offset):
    import torch
    dt = np.uint16 if ol.PF_WIDE[pf] else np.uint8
    rows, cols = ol.frame_shape(pf, w, h)
    buf = np.random.RandomState(w).randint(0, 1024 if ol.PF_WIDE[pf] else 256, (rows, cols)).astype(dt)
    frame, out = Placed((rows, cols), dt, 0, 0, device, buf), Placed((h, w, 3), np.float32, offset, 0, device)
    cases.yuv_to_rgb(pf, cr, cp, frame.view(), w, h, out.view())
    torch.cuda.synchronize()
    assert out.read().tobytes() == ol.oracle_yuv_to_rgb(pf, cr, cp, buf, w, h).tobytes()


@pytest.mark.parametrize("pf,cr,cp", [(ol.PF_NV12, 0, 1), (ol.PF_NV21, 1, 0), (ol.PF_P010, 0, 2), (ol.PF_UYVY, 1, 2)])
@pytest.mark.parametrize("w,h", [(2050, 1000), (2047, 1001), (1922, 1080)])
def test_line_aligned_segments_rgb_to_video(device, pf, cr, cp, w, h):
    import torch
    dt = np.uint16 if ol.PF_WIDE[pf] else np.uint8
    rgb = np.random.RandomState(w).randint(0, 1024 if ol.PF_WIDE[pf] else 256, (h, w, 3)).astype(dt)
    rows, cols = ol.frame_shape(pf, w + (w & 1), h + (h & 1))
    if pf in (ol.PF_NV12, ol.PF_NV21, ol.PF_P010):
        rows = h + (h + 1) // 2
    start = np.full((rows, cols), 9, dt)
    frame, src = Placed((rows, cols), dt, 0, 0, device, start), Placed((h, w, 3), dt, 0, 0, device, rgb)
    cases.rgb_to_yuv(pf, cr, cp, src.view(), frame.view())
    torch.cuda.synchronize()
    assert np.array_equal(frame.read(), ol.oracle_rgb_to_yuv(pf, cr, cp, rgb, start))


@pytest.mark.parametrize("w,h,offset", [(961, 2101, 4), (1025, 2000, 8)])
def test_line_aligned_segments_warp(device, w, h, offset):
    import torch
    img = np.random.RandomState(w).randint(0, 256, (h, w, 3)).astype(np.uint8)
    m = np.array([[0.99, -0.12, 4.5], [0.12, 0.99, -3.25]], np.float32)
    out = Placed((h, w, 3), np.float32, offset, 0, device)
    cases.warp(torch.from_numpy(img).to(device), m, False, (w, h), out.view())
    torch.cuda.synchronize()
    assert out.read().tobytes() == ol.oracle_warp(img, 3, m, (w, h), False).tobytes()


# Whole lines (rows of 2 048 elements: the grid has a column of workgroups more than the row alone needs) and half lines, for every
# size class of elements, in a tensor whose planes are no whole lines apart, so that each plane's rows have phases of their own
# (or none: elements of more than one sample whose rows never meet a line boundary in the planes after the first).
# Element sizes 1, 2, 3, 6 leave a row's ends element by element, 4 as runs, 8 (ushort4, float2), 12 and 16 through the LDS, 8
# (double), 24 and 32 as runs again.
@pytest.mark.parametrize("kind", range(len(cases.TENSOR_KINDS)))
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("in_place", [False, True])
def test_line_aligned_segments_tensors(device, kind, half, in_place):
    import torch
    from fusedkernellibrary_amd import last_launch
    base, cn = cases.TENSOR_KINDS[kind]
    size, planes = np.dtype(base).itemsize, 3
    elem = size * cn
    unit = elem & -elem                                            # the power of two in an element's size
    half_line = 128 // unit // 2 - 1                               # elements that a row's first segment begins left of it, at most
    w = 1024 - half_line if half else 2048                         # four segments with half lines, five with whole ones
    h = (16000000 if elem % 4 else 24000000) // (w * elem * planes) + 1
    rng = np.random.RandomState(kind)
    row, data = w * elem, rng.randint(0, 256, (planes, h, w * elem)).astype(np.uint8)

    def place(offset, pad, plane_pad, fill):
        pitches = (row + pad, (row + pad) * h + plane_pad)
        host = np.full(256 + offset + pitches[1] * planes + 256, FILL, np.uint8)
        at = np.lib.stride_tricks.as_strided(host[256 + offset:], (planes, h, row), (pitches[1], pitches[0], 1))
        if fill:
            at[:] = data
        return host, at, pitches, 256 + offset

    out_host, out_at, out_pitches, out_start = place(3 * unit, unit * (kind % 3 + 1), 5 * size, in_place)
    out = torch.from_numpy(out_host).to(device)
    if in_place:
        cases.copy_tensor(kind, out[out_start:], out_pitches, out[out_start:], out_pitches, w, h, planes)
    else:
        src_host, _, src_pitches, src_start = place(size, 0, size, True)
        cases.copy_tensor(kind, torch.from_numpy(src_host).to(device)[src_start:], src_pitches, out[out_start:], out_pitches, w, h, planes)
    torch.cuda.synchronize()
    assert last_launch()["grid"][0] == (4 if half else 9)
    out_at[:] = data
    assert np.array_equal(out.cpu().numpy(), out_host)             # the rows are the input's, every byte beside them is as it was


# Launches that write up to 4 MiB store without the non-temporal hint, larger ones with it: both sides of
# the line, in widths below those of line-aligned segments, whole runs and remainders.
@pytest.mark.parametrize("w,h", [(300, 1165), (300, 1166), (299, 1168), (299, 1170), (301, 1161), (301, 1162)])
def test_small_and_larger_outputs(device, w, h):
    import torch
    rng = np.random.RandomState(w + h)
    mul, add = rng.uniform(0.5, 2.0, (4, 3)).astype(np.float32), rng.uniform(-64, 64, (4, 3)).astype(np.float32)
    imgs = [rng.randint(0, 256, (h, w, 3)).astype(np.uint8) for _ in range(4)]                   # 4 194 000 ... 4 197 600 bytes
    srcs = [Placed((h, w, 3), np.uint8, 0, 0, device, a) for a in imgs]
    outs = [Placed((h, w, 3), np.uint8, 0, 0, device) for _ in imgs]
    cases.batch_muladd_sat([s.view() for s in srcs], mul, add, [o.view() for o in outs])
    fh = 3 * h                                                                                 # as many bytes of floats
    img = rng.uniform(-1, 1, (fh, w)).astype(np.float32)
    src, out = Placed((fh, w), np.float32, 4, 0, device, img), Placed((fh, w), np.float32, 8, 0, device)
    cases.add_mul_chain(src.view(), 3, 0.5, 1.0001, out.view())
    padded = torch.zeros((4 * h, w, 3), dtype=torch.uint8, device=device)                      # a kernel for whole runs only
    cases.pad(srcs[0].view(), ol.BORDER_REFLECT_101, 8, 8, padded)
    torch.cuda.synchronize()
    for b, c in zip(outs, ol.oracle_batch_muladd_sat(imgs, mul, add)):
        assert np.array_equal(b.read(), c)
    assert out.read().tobytes() == ol.oracle_add_mul_chain(img, 3, np.float32(0.5), np.float32(1.0001)).tobytes()
    assert padded.cpu().numpy().tobytes() == ol.oracle_pad(imgs[0], ol.BORDER_REFLECT_101, 8, 8, w, 4 * h).tobytes()


@pytest.mark.parametrize("pf,cr,cp", [(ol.PF_NV12, 0, 1), (ol.PF_P010, 0, 2), (ol.PF_UYVY, 1, 1)])
@pytest.mark.parametrize("w,h", [(300, 1164), (300, 1166), (254, 1376), (258, 1356)])
def test_small_and_larger_video_frames(device, pf, cr, cp, w, h):
    """Decoded to float3 and encoded from RGB, as many bytes stored: chains compiled ahead of time and on first use."""
    import torch
    dt, size = (np.uint16, 2) if ol.PF_WIDE[pf] else (np.uint8, 1)
    rng = np.random.RandomState(w + pf)
    rows, cols = ol.frame_shape(pf, w, h)
    buf = rng.randint(0, 1024 if size == 2 else 256, (rows, cols)).astype(dt)
    frame, out = Placed((rows, cols), dt, 0, 0, device, buf), Placed((h, w, 3), np.float32, 4, 0, device)
    cases.yuv_to_rgb(pf, cr, cp, frame.view(), w, h, out.view())
    eh = {ol.PF_NV12: 8, ol.PF_P010: 4, ol.PF_UYVY: 6}[pf] * h                                 # 1.5, 3 and 2 bytes a pixel instead of 12
    rgb = rng.randint(0, 1024 if size == 2 else 256, (eh, w, 3)).astype(dt)
    rows, cols = ol.frame_shape(pf, w, eh)
    start = np.full((rows, cols), 9, dt)
    encoded, src = Placed((rows, cols), dt, 0, 0, device, start), Placed((eh, w, 3), dt, 0, 0, device, rgb)
    cases.rgb_to_yuv(pf, cr, {ol.PF_UYVY: 2}.get(pf, cp), src.view(), encoded.view())
    torch.cuda.synchronize()
    assert out.read().tobytes() == ol.oracle_yuv_to_rgb(pf, cr, cp, buf, w, h).tobytes()
    assert np.array_equal(encoded.read(), ol.oracle_rgb_to_yuv(pf, cr, {ol.PF_UYVY: 2}.get(pf, cp), rgb, start))


@pytest.mark.parametrize("pf,cr,cp", [(ol.PF_NV12, 0, 1), (ol.PF_NV21, 0, 0), (ol.PF_P010, 0, 2)])
def test_video_frames_of_odd_width_to_rgb(device, pf, cr, cp):
    """The last four pixels of a row of odd width begin inside a chroma pair."""
    import torch
    dt = np.uint16 if ol.PF_WIDE[pf] else np.uint8
    rng = np.random.RandomState(170 + pf)
    for n, w in enumerate((1, 3, 5, 7, 9, 255, 257, 259, 511, 515, 1021)):
        h = (2, 6, 12)[n % 3]
        rows, cols = ol.frame_shape(pf, w + 1, h)
        buf = rng.randint(0, 1024 if ol.PF_WIDE[pf] else 256, (rows, cols)).astype(dt)
        frame, out = Placed((rows, cols), dt, 0, 0, device, buf), Placed((h, w, 3), np.float32, 4, 4, device)
        cases.yuv_to_rgb(pf, cr, cp, frame.view(), w, h, out.view())
        torch.cuda.synchronize()
        assert out.read().tobytes() == ol.oracle_yuv_to_rgb(pf, cr, cp, buf, w + 1, h)[:, :w].tobytes(), (w, h)
