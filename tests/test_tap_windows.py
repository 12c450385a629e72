"""Which bytes the bilinear kernels' tap accesses touch, worked out on the CPU for small, tight-pitch, odd-aligned images.

The kernels fetch the two horizontally adjacent taps of a pixel as ONE dword-aligned window: it starts at the dword
boundary at or below the first tap and is 12 bytes long for 3-byte pixels (include/fkd/ops.hpp, PairWindow), so it can
reach up to 6 bytes past the second tap.  Two rules keep that inside the allocation, and torch's padded allocations
would hide a violation on the GPU, so they are checked here by brute force over every tap position:

* tile form (k_gather): waves whose taps reach a row with (height - 1 - y) * pitch < 8 bytes of image behind its start
  take one access per channel instead (Read2D::tap_row / tap_last); every other window must end inside the image;
* strip form (k_strip): the buffer resource ends with the dword that holds the image's last byte (make_tap_image with a
  size); dwords at or beyond that extent are not fetched (they read as zero).  Every byte a blend USES must lie in a
  delivered dword, and every delivered dword must start inside the image, so that it lies in a mapped page.  Warps fetch the same
  way.
"""
import ctypes as C
import itertools

import pytest

import fkl_cases as cases

ELEM = 3          # bytes per pixel (uchar3)
WINDOW = 12       # dwords fetched per pair window: 3


def _image_bytes(w, h, pitch):
    return pitch * (h - 1) + w * ELEM


def _cases():
    for w, h in itertools.product((2, 3, 5, 8, 11), (1, 2, 3, 5)):
        for pad in (0, 1, 2, 3, 5):
            for lo in (0, 1, 2, 3):               # offset of the image's first byte inside its dword
                yield w, h, w * ELEM + pad, lo


def test_tile_form_windows_stay_inside_the_image():
    checked = 0
    for w, h, pitch, lo in _cases():
        size = _image_bytes(w, h, pitch)
        for y in range(h):
            last = (h - 1 - y) * pitch < 8                      # Read2D::tap_row
            for x1 in range(w - 1):                             # first tap; the second one is x1 + 1 <= w - 1
                first_byte = y * pitch + x1 * ELEM              # relative to the image's first byte
                if last:
                    touched = range(first_byte, first_byte + 2 * ELEM)          # channel by channel, nothing else
                else:
                    start = ((lo + first_byte) & ~3) - lo       # the dword at or below the first tap (rows of any alignment)
                    touched = range(start, start + WINDOW)
                    # a window may begin up to 3 bytes before its first tap: the same dword as a byte that is needed
                    assert first_byte - start <= 3
                assert touched[-1] < size, (w, h, pitch, lo, y, x1)
                assert touched[0] >= -3                         # at most the image's own first dword
                checked += 1
    assert checked > 5000


# samples of 1, 2 and 4 bytes: an image's rows start and repeat at multiples of their samples' size
@pytest.mark.parametrize("elem,sample", [(1, 1), (2, 1), (3, 1), (4, 1), (6, 2), (8, 4)])
def test_strip_form_windows_hold_every_used_byte_and_touch_nothing_unmapped(elem, sample):
    """The library's own window arithmetic (fkd::detail::pair_window_at, tap_extent), compiled for the host: strip form and warps,
    images of every address and pitch."""
    window_of = cases.cases().fklcase_tap_window
    out = (C.c_uint * 4)()
    checked = 0
    for w, h in itertools.product((2, 3, 5, 8, 11), (1, 2, 3, 5)):
        for pad, lo in itertools.product(range(0, 6, sample), range(0, 4, sample)):
            pitch = w * elem + pad
            size = pitch * (h - 1) + w * elem
            for y, x1 in itertools.product(range(h), range(w - 1)):
                at = lo + x1 * elem + y * pitch                     # from the dword at or below the image's first byte
                assert window_of(elem, at, size, lo, out) == 0
                start, drop, length, extent = out
                assert extent % 4 == 0 and extent - 4 < lo + size   # every delivered dword starts inside the image: a mapped page
                assert start + drop == at and drop + 2 * elem <= length         # the pair is where it is looked for
                assert at + 2 * elem <= extent                      # and all of it is delivered
                if elem % 4:
                    assert start % 4 == 0 and drop <= 3 and start <= extent - 4
                else:
                    assert drop == 0 and length == 2 * elem
                checked += 1
    assert checked > 500


def test_columns_without_a_window_touch_no_image():
    """The strip form marks a column beyond the output with the offset 2 GB; with any row's offset on top it is beyond the extent of
    the largest image the form takes, and does not wrap."""
    largest = 0x7ffffff0 - 1
    out = (C.c_uint * 4)()
    for elem, row, lo in itertools.product((1, 2, 3, 4, 6, 8), (0, 1, 2, 3, 4097, largest), range(4)):
        assert cases.cases().fklcase_tap_window(elem, 0x80000000 + row, largest, lo, out) == 0
        assert out[0] >= 0x80000000 > out[3] and out[0] + out[2] <= 0xffffffff


@pytest.mark.parametrize("kind", range(5))
def test_warps_look_for_a_rectangles_rows_where_the_image_has_them(kind):
    """A warp's row offset is the first row's plus whole pitches (fkd::Warp::tap_row): rectangles at and off the image's top, with operations on
    either side, for pitches up to the 24 bits the multiplication takes."""
    out = (C.c_uint * 3)()
    for pitch, top, height in itertools.product((6, 1920, 5763, 0xfffffd), (0, 1, 20, 77), (1, 2, 100)):
        for y in (0, 1, height // 2, height - 1):
            assert cases.cases().fklcase_warp_tap_row(kind, pitch, top, height, y, out) == 0
            assert out[2] == 1 and out[0] == out[1] % (1 << 32), (pitch, top, y)
    assert cases.cases().fklcase_warp_tap_row(kind, 1 << 24, 1, 10, 0, out) == 0 and out[2] == 0
    assert cases.cases().fklcase_warp_tap_row(kind, 6, 1, 1 << 24, 0, out) == 0 and out[2] == 0
