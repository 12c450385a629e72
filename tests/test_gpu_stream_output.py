"""Planar outputs of the bilinear kernel on both sides of the size from which they are stored past the last-level cache
(80 MiB): the two kinds of store leave the same bytes, the oracle's, in both forms of the kernel and in a chain compiled on
first use."""
import numpy as np
import pytest

import fkl_cases as cases
import oracle_lib as ol
import workloads as wl
from fusedkernellibrary_amd import last_launch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dst,kernel", [((293, 372), None), ((293, 373), None),      # 83 708 928 and 83 933 952 bytes: ragged rows
                                        ((251, 435), "gather"), ((251, 436), "gather"),
                                        ((224, 487), "strip"), ((224, 488), "strip")])     # 83 779 584 and 83 951 616 bytes: rows of whole lines
def test_batches_around_the_limit(dst, kernel):
    import torch
    c = wl.config3(width=640 if kernel else 641, height=359, min_side=2, span=340)      # rows that share their alignment, or not
    src = torch.from_numpy(c["src"]).cuda()
    out = torch.full((64, 3, dst[1], dst[0]), -7.0, dtype=torch.float32, device="cuda")
    cases.crop_resize_norm_split(src, c["rects"], dst, c["sub"], c["div"], out)
    torch.cuda.synchronize()
    if kernel:
        assert last_launch()["kernel"] == kernel
    want = ol.oracle_crop_resize_norm_split(c["src"], c["rects"], dst, c["sub"], c["div"])
    assert out.cpu().numpy().tobytes() == want.tobytes()


@pytest.mark.parametrize("dst,offset,kernel", [((224, 512), 0, "strip"), ((224, 512), 32, "strip"), ((224, 512), 16, "gather"),
                                               ((224, 512), 1, "gather"), ((48, 2390), 0, "strip"), ((48, 2390), 8, "gather"), ((31, 3700), 0, "strip")])
def test_outputs_on_and_off_the_lines(dst, offset, kernel):
    """An output that begins `offset` floats after a line boundary: its rows are whole lines, whole half lines or neither."""
    import torch
    c = wl.config3(width=640, height=359, min_side=2, span=340)
    src = torch.from_numpy(c["src"]).cuda()
    n = 64 * 3 * dst[0] * dst[1]
    buf = torch.full((n + 64,), -7.0, dtype=torch.float32, device="cuda")
    assert buf.data_ptr() % 128 == 0
    cases.crop_resize_norm_split(src, c["rects"], dst, c["sub"], c["div"], buf[offset:offset + n].view(64, 3, dst[1], dst[0]))
    torch.cuda.synchronize()
    assert last_launch()["kernel"] == kernel
    got = buf.cpu().numpy()
    assert (got[:offset] == -7.0).all() and (got[offset + n:] == -7.0).all()
    assert got[offset:offset + n].tobytes() == ol.oracle_crop_resize_norm_split(c["src"], c["rects"], dst, c["sub"], c["div"]).tobytes()


@pytest.mark.parametrize("dst", [(1526, 1526), (1527, 1527), (201, 11593)])          # 83 832 336, 83 942 244 and 83 886 948 bytes
def test_a_chain_compiled_on_first_use(dst):
    import torch
    rng = np.random.RandomState(11)
    img = rng.randint(0, 256, (200, 320, 3)).astype(np.uint8)
    rects = np.array([[10, 20, 300, 60], [40, 0, 50, 200], [100, 50, 120, 120]], np.int32)
    bg, mul = np.array([0.25, 128.5, 255.0], np.float32), np.array([0.5, 2.0, 1.0 / 255.0], np.float32)
    out = torch.full((3, 3, dst[1], dst[0]), -7.0, dtype=torch.float32, device="cuda")
    cases.uncompiled_letterbox_split_b3(torch.from_numpy(img).cuda(), rects, dst, bg, mul, out)
    torch.cuda.synchronize()
    want = np.zeros((3, 3, dst[1], dst[0]), np.float32)
    reads = [ol.read_2d(img, 3, crop=rects[i], resize=dst, ar=ol.PRESERVE_AR, bg=tuple(bg) + (0.0,)) for i in range(3)]
    ol.execute(reads, [ol.op(ol.MUL, tuple(mul) + (0.0,))], [ol.write(ol.TENSOR_SPLIT, want, 3, dst[0], dst[1], 3, 3)])
    assert out.cpu().numpy().tobytes() == want.tobytes()
