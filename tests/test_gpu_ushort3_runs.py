"""Runs of four ushort3 (24 bytes, two accesses): 10-bit RGB to P010 at every address and pitch that leaves the samples aligned, for widths around
runs, waves and segments, bit for bit the oracle's.  (Copies of such images: test_gpu_any_alignment, test_gpu_flat_planes.)"""
import numpy as np
import pytest

import fkl_cases as cases
import oracle_lib as ol
from test_gpu_any_alignment import Placed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offset", [0, 2])
@pytest.mark.parametrize("pad", [0, 2, 4])
def test_rgb_to_p010(device, offset, pad):
    import torch
    for n, (w, h) in enumerate(((2, 2), (4, 4), (6, 2), (10, 6), (130, 4), (254, 2), (256, 10), (258, 4), (514, 2), (1022, 4), (1280, 722))):
        rgb = np.random.RandomState(n).randint(0, 1024, (h, w, 3)).astype(np.uint16)
        src = Placed(rgb.shape, np.uint16, offset, pad, device, rgb)
        out = Placed((h * 3 // 2, w), np.uint16, offset, pad, device)
        cases.rgb_to_yuv(ol.PF_P010, 0, 2, src.view(), out.view())
        torch.cuda.synchronize()
        want = np.zeros((h * 3 // 2, w), np.uint16)
        ol.oracle_rgb_to_yuv(ol.PF_P010, 0, 2, rgb, want)
        assert np.array_equal(out.read(), want), (w, h)
