"""How many rows a thread of the rows kernel takes (fkd::rows_halved): the grids of chains that keep all their rows where those make a round of
two to four workgroups per compute unit, on both sides of either end, and the results, which do not depend on it."""
import numpy as np
import pytest

import oracle_lib as ol
from fusedkernellibrary_amd import last_launch
import fkl_cases as cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pf", [ol.PF_NV12, ol.PF_P010])
@pytest.mark.parametrize("w,h,rows", [(1026, 814, 1), (1026, 820, 2), (1538, 1168, 2), (1538, 1178, 1)])
def test_decoders(device, pf, w, h, rows):
    import torch
    dt = np.uint16 if ol.PF_WIDE[pf] else np.uint8
    frame = np.random.default_rng(61).integers(0, 1024 if ol.PF_WIDE[pf] else 256, ol.frame_shape(pf, w, h)).astype(dt)
    out = torch.full((h, w, 3), -7.0, dtype=torch.float32, device=device)
    cases.yuv_to_rgb(pf, 0, 1 if pf == ol.PF_NV12 else 2, torch.from_numpy(frame.view(np.int16) if ol.PF_WIDE[pf] else frame).to(device), w, h, out)
    torch.cuda.synchronize()
    assert last_launch()["grid"] == [-(-w // 256), -(-h // (4 * rows)), 1]
    assert out.cpu().numpy().tobytes() == ol.oracle_yuv_to_rgb(pf, 0, 1 if pf == ol.PF_NV12 else 2, frame, w, h).tobytes()


@pytest.mark.parametrize("gap", [0, 1])
@pytest.mark.parametrize("w,h,rows", [(768, 1360, 1), (768, 1366, 2), (768, 2720, 2), (768, 2740, 1)])
def test_elements_exchanged_at_both_ends(device, w, h, rows, gap):
    import torch
    src = torch.randn((h, w + gap, 3), device=device)
    out = torch.zeros((h, w, 3), device=device)
    cases.pointwise(0, src.view(torch.uint8).view(h, -1), w, h, out.view(torch.uint8).view(h, -1))
    torch.cuda.synchronize()
    launch = last_launch()
    assert launch["form"] == ("rows" if gap else "flat")
    if gap: assert launch["grid"] == [3, -(-h // (4 * rows)), 1]
    else: assert launch["grid"][0] in (-(-w * h // (1024 * rows)), -(-(w * h + 31) // (1024 * rows)))
    assert torch.equal(out, src[:, :w].abs())
