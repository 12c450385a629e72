"""Which form of the bilinear kernel a launch takes (fkd::strip_pays, compiled for the host): launches that were measured clearly
on one side, and the alignment of output rows that the rule asks for.  That both forms give the same result whatever the rule says is
tested elsewhere."""
import pytest

import fkl_cases as cases


@pytest.mark.parametrize("address,w,h,planes,grain", [
    (0x7f0000000000, 224, 224, 64, 128), (0x7f0000000000, 640, 640, 1, 128), (0x7f0000000000, 240, 520, 64, 64),
    (0x7f0000000000, 200, 625, 64, 32), (0x7f0000000000, 100, 1250, 64, 16), (0x7f0000000000, 225, 225, 64, 4),
    (0x7f0000000004, 224, 640, 64, 4), (0x7f0000000020, 224, 640, 64, 32), (0x7f0000000040, 224, 640, 64, 64),
    (0x7f0000000080, 224, 640, 64, 128)])
def test_alignment_of_output_rows(address, w, h, planes, grain):
    assert cases.cases().fklcase_row_grain(address, w, h, planes) == grain


@pytest.mark.parametrize("w,h,planes,any_pitch,grain,strip", [
    # outputs stored past the last-level cache
    (224, 1280, 64, False, 128, True), (224, 1280, 64, False, 4, False), (224, 1280, 64, False, 64, False), (160, 781, 64, True, 128, True),
    (48, 2343, 64, False, 64, True), (48, 2343, 64, False, 32, False), (144, 976, 64, True, 64, True), (240, 1302, 64, False, 64, False),
    (28, 4017, 64, False, 16, True), (20, 5625, 64, True, 16, True), (60, 1875, 64, False, 16, False), (100, 1250, 64, False, 16, False),
    (200, 1092, 64, False, 32, False), (225, 1274, 64, True, 4, False),
    # smaller ones: images whose rows share their alignment
    (224, 224, 64, False, 128, True), (100, 200, 64, False, 16, True), (200, 406, 64, False, 32, True), (165, 170, 64, False, 4, True),
    (165, 378, 64, False, 4, False), (180, 156, 64, False, 16, True), (180, 277, 64, False, 16, False), (197, 79, 64, False, 4, True), (197, 253, 64, False, 4, False),
    (212, 132, 64, False, 16, True), (212, 383, 64, False, 16, False), (225, 83, 64, False, 4, True), (225, 222, 64, False, 4, False),
    (252, 86, 64, False, 16, True), (236, 211, 64, False, 16, False), (250, 800, 8, False, 8, False),
    # ... and images whose rows do not
    (160, 200, 64, True, 128, True), (224, 224, 64, True, 128, True), (200, 60, 8, True, 32, False), (225, 60, 64, True, 4, False),
    (105, 119, 64, True, 4, True), (125, 437, 64, True, 4, False), (112, 279, 64, True, 64, True), (130, 300, 64, True, 8, True),
    (64, 39, 8, True, 128, False), (64, 156, 8, True, 128, True)])
def test_form_of_measured_launches(w, h, planes, any_pitch, grain, strip):
    assert cases.cases().fklcase_strip_pays(w, h, planes, int(any_pitch), grain) == int(strip)
