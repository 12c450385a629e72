"""The work a program has this library do, as measurable cases: fused image chains through the C++ host API.

Every case takes one image, frame or batch through a chain spelled with executeOperations<TransformDPP<>> (the chains of
tests/cases/fkl_cases.cpp, built into libfkl_cases.so), with device memory the caller owns, on the caller's stream, without a
synchronisation.  A pass over small images takes several of them ("frames"), one call each, as a program with several cameras
or a folder of pictures does.  Eight kinds of chain, each with the range of sizes that real programs bring to it:

  thumbs     5 crops of one image -> letterboxed thumbnails (PRESERVE_AR) -> mul, sub, saturate -> uint8 tensor
  crops      8 or 64 crops of one image -> bilinear resize -> BGR2RGB -> (x - mean) / std -> planar float tensor
  chain      one float image through n additions and multiplications
  images     4 or 100 separate uint8 images, per-image mul and add, saturated back to uint8
  nv12       NV12 video frame -> RGB -> bilinear resize -> scale -> planar float tensor
  encode     RGB image -> YUV -> saturate -> video frame (NV12, P010 or UYVY)
  decode     video frame (NV12, P010 or UYVY) -> RGB float image
  warp       affine or perspective warp of a uint8 image into a float image

Images are tightly packed, as decoders hand them over: an odd width makes 3-byte rows that start at every byte alignment.
Pixels are uniform random (the chains' work does not depend on them); crop rectangles and per-image factors are drawn from the
same seed.  The library's results are defined bit by bit (one rounding per operation, in the chain's order), so every output
has to stay exactly the same.
"""
import ctypes as C
import functools
import math
import os
import random

import numpy as np
import torch

import fusedkernellibrary_amd as fkl

NV12, P010, UYVY = 0, 3, 10          # fk::PixelFormat
# (ColorRange, ColorPrimitives) the chains are spelled with: full / limited and bt601 / bt709 / bt2020
ENCODE_AS = {NV12: (0, 1), P010: (0, 2), UYVY: (1, 2)}
DECODE_AS = {NV12: (0, 1), P010: (0, 2), UYVY: (1, 1)}
CHAIN_LENGTHS = (1, 2, 3, 10, 20, 30, 40, 50, 100)
MEAN = [255.0 * v for v in (0.485, 0.456, 0.406)]
STD = [255.0 * v for v in (0.229, 0.224, 0.225)]


def listed():
    return [
        # the README program on four cameras: five small regions of a 4K image as 128x64 thumbnails; latency of small calls
        {"name": "thumbs_5x128x64", "kind": "thumbs", "frames": 4, "w": 3840, "h": 2160, "dw": 128, "dh": 64, "lo": 16, "hi": 140},
        # a handful of detections in each of four photographs (rows of 1279 * 3 bytes start at every alignment) for a classifier
        {"name": "crops_8x224_photo", "kind": "crops", "frames": 4, "batch": 8, "w": 1279, "h": 853, "dw": 224, "dh": 224, "lo": 64, "hi": 512},
        # the headline workload: 64 crops of a 1080p frame as one classifier batch
        {"name": "crops_64x224", "kind": "crops", "batch": 64, "w": 1920, "h": 1080, "dw": 224, "dh": 224, "lo": 64, "hi": 512},
        # 64 tiles of a 4K frame for a detector's 640x640 input: wide outputs
        {"name": "crops_64x640", "kind": "crops", "batch": 64, "w": 3840, "h": 2160, "dw": 640, "dh": 640, "lo": 320, "hi": 1280},
        # vertical fusion: a 4K float image through 50 arithmetic operations in one pass
        {"name": "chain_50_2160p", "kind": "chain", "n": 50, "w": 3840, "h": 2160},
        # horizontal fusion: brightness and contrast of a batch of four images of odd size ...
        {"name": "images_4_odd", "kind": "images", "batch": 4, "w": 1279, "h": 719},
        # ... and of a hundred 1080p images, the largest call
        {"name": "images_100_1080p", "kind": "images", "batch": 100, "w": 1920, "h": 1080},
        # video to network: a 4K frame halved in both directions ...
        {"name": "nv12_2160p_to_1080p", "kind": "nv12", "w": 3840, "h": 2160, "dw": 1920, "dh": 1080},
        # ... and a 1080p frame to a detector's 1333x800, by factors that are not whole
        {"name": "nv12_1080p_to_1333x800", "kind": "nv12", "w": 1920, "h": 1080, "dw": 1333, "dh": 800},
        # rendered RGB frame to a video encoder's input
        {"name": "encode_nv12_2160p", "kind": "encode", "pf": NV12, "w": 3840, "h": 2160},
        # capture card (packed 4:2:2) to RGB
        {"name": "decode_uyvy_2160p", "kind": "decode", "pf": UYVY, "w": 3840, "h": 2160},
        # image registration: a 4K image turned by 7 degrees
        {"name": "warp_affine_2160p", "kind": "warp", "perspective": False, "w": 3840, "h": 2160, "angle": 7.0, "zoom": 1.0},
    ]


def _log(rng, lo, hi, even=False):
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(2, v & ~1) if even else v


def draw(rng):
    case = _draw(rng)
    # small images come several at a time
    if case.get("batch") != 100 and _work_per_frame(case)["bytes"] < 24e6:
        case["frames"] = 4
    return case


def _draw(rng):
    kind = rng.choice(["thumbs", "crops", "crops", "chain", "images", "images", "nv12", "nv12", "encode", "decode", "warp"])
    if kind == "thumbs":
        w, h = _log(rng, 320, 3840), _log(rng, 180, 2160)
        return {"kind": kind, "w": w, "h": h, "dw": _log(rng, 32, 256), "dh": _log(rng, 32, 256), "lo": 16, "hi": rng.randint(64, min(w, h))}
    if kind == "crops":
        w, h = _log(rng, 320, 3840), _log(rng, 180, 2160)
        return {"kind": kind, "batch": rng.choice([8, 64]), "w": w, "h": h, "dw": _log(rng, 64, 640), "dh": _log(rng, 64, 640),
                "lo": 32, "hi": rng.randint(64, min(w, h))}
    if kind == "chain":
        return {"kind": kind, "n": rng.choice(CHAIN_LENGTHS), "w": _log(rng, 64, 3840), "h": _log(rng, 36, 2160)}
    if kind == "images":
        return {"kind": kind, "batch": rng.choice([4, 100]), "w": _log(rng, 64, 1920), "h": _log(rng, 36, 1080)}
    if kind == "nv12":
        return {"kind": kind, "w": _log(rng, 320, 3840, even=True), "h": _log(rng, 180, 2160, even=True), "dw": _log(rng, 64, 1920),
                "dh": _log(rng, 64, 1080)}
    if kind == "encode" or kind == "decode":
        return {"kind": kind, "pf": rng.choice([NV12, P010, UYVY]), "w": _log(rng, 128, 3840, even=True), "h": _log(rng, 72, 2160, even=True)}
    return {"kind": kind, "perspective": rng.random() < 0.3, "w": _log(rng, 128, 3840), "h": _log(rng, 72, 2160),
            "angle": round(rng.uniform(-30.0, 30.0), 2), "zoom": round(rng.uniform(0.6, 1.6), 3)}


@functools.lru_cache(maxsize=None)
def _library():
    fkl.lib()
    return C.CDLL(os.path.join(fkl.ROOT_DIR, "tests", "cases", "libfkl_cases.so"))


def _ptr(x):
    return C.c_void_p(x.data_ptr() if isinstance(x, torch.Tensor) else x.ctypes.data)


def _rects(rng, n, case):
    """n crop rectangles (x, y, w, h) inside the image, their sides between case["lo"] and case["hi"] pixels."""
    out = np.zeros((n, 4), np.int32)
    for i in range(n):
        w = min(rng.randint(case["lo"], case["hi"]), case["w"])
        h = min(rng.randint(case["lo"], case["hi"]), case["h"])
        out[i] = (rng.randint(0, case["w"] - w), rng.randint(0, case["h"] - h), w, h)
    return out


def _frame_shape(pf, w, h):
    """Rows and samples per row of a w x h frame in pixel format pf."""
    return (h, 2 * w) if pf == UYVY else (h * 3 // 2, w)


def prepare(case, seed):
    rng = random.Random(seed)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(rng.getrandbits(40))
    frames = [_prepare_frame(case, rng, gen) for _ in range(case.get("frames", 1))]
    return {"calls": [f[0] for f in frames], "outs": [f[1] for f in frames], "keep": [f[2] for f in frames]}


def _prepare_frame(case, rng, gen):
    """(the bound call, its output, what has to stay alive with it) for one image, frame or batch."""
    lib = _library()
    kind, w, h = case["kind"], case["w"], case["h"]

    def pixels(*shape, top=256, dtype=torch.uint8):
        return torch.randint(0, top, shape, dtype=dtype, device="cuda", generator=gen)

    def output(*shape, dtype=torch.float32):
        return torch.zeros(shape, dtype=dtype, device="cuda")

    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    if kind == "thumbs":
        src, out = pixels(h, w, 3), output(5, case["dh"], case["dw"], 3, dtype=torch.uint8)
        keep = [src, _rects(rng, 5, case), np.zeros(3, np.float32), np.full(3, 2.0, np.float32), np.full(3, 128.0, np.float32)]
        args = [stream, _ptr(src), w, h, 3 * w, _ptr(keep[1]), case["dw"], case["dh"], _ptr(keep[2]), _ptr(keep[3]), _ptr(keep[4]), _ptr(out)]
        fn = lib.fklcase_crop_resize_par_u8_b5
    elif kind == "crops":
        b = case["batch"]
        src, out = pixels(h, w, 3), output(b, 3, case["dh"], case["dw"])
        keep = [src, _rects(rng, b, case), np.array(MEAN, np.float32), np.array(STD, np.float32)]
        args = [stream, _ptr(src), w, h, 3 * w, _ptr(keep[1]), case["dw"], case["dh"], _ptr(keep[2]), _ptr(keep[3]), _ptr(out)]
        fn = {8: lib.fklcase_crop_resize_norm_split_b8, 64: lib.fklcase_crop_resize_norm_split_b64}[b]
    elif kind == "chain":
        src, out = torch.rand((h, w), device="cuda", generator=gen) * 2 - 1, output(h, w)
        keep = [src]
        args = [stream, _ptr(src), w, h, 4 * w, case["n"], C.c_float(0.5), C.c_float(1.0001), _ptr(out), 4 * w, 0]
        fn = lib.fklcase_add_mul_chain
    elif kind == "images":
        b = case["batch"]
        srcs, out = [pixels(h, w, 3) for _ in range(b)], output(b, h, w, 3, dtype=torch.uint8)
        mul = np.array([[rng.uniform(0.5, 2.0) for _ in range(3)] for _ in range(b)], np.float32)
        add = np.array([[rng.uniform(-64.0, 64.0) for _ in range(3)] for _ in range(b)], np.float32)
        ins = (C.c_void_p * b)(*[s.data_ptr() for s in srcs])
        outs = (C.c_void_p * b)(*[out.data_ptr() + i * h * w * 3 for i in range(b)])
        keep = [srcs, mul, add, ins, outs]
        args = [stream, ins, w, h, 3 * w, _ptr(mul), _ptr(add), outs, 3 * w]
        fn = {4: lib.fklcase_batch_muladd_sat_b4, 100: lib.fklcase_batch_muladd_sat_b100}[b]
    elif kind == "nv12":
        src, out = pixels(*_frame_shape(NV12, w, h)), output(3, case["dh"], case["dw"])
        keep = [src]
        args = [stream, _ptr(src), w, h, w, case["dw"], case["dh"], C.c_float(1.0 / 255.0), _ptr(out)]
        fn = lib.fklcase_nv12_rgb_resize_split
    elif kind == "encode" or kind == "decode":
        pf = case["pf"]
        size, kind_of = (2, {"top": 1024, "dtype": torch.int16}) if pf == P010 else (1, {})
        shape = _frame_shape(pf, w, h)
        if kind == "encode":
            src, out = pixels(h, w, 3, **kind_of), output(*shape, dtype=torch.int16 if pf == P010 else torch.uint8)
            args = [stream, pf, *ENCODE_AS[pf], _ptr(src), w, h, 3 * w * size, _ptr(out), shape[1] * size]
            fn = lib.fklcase_rgb_to_yuv
        else:
            src, out = pixels(*shape, **kind_of), output(h, w, 3)
            args = [stream, pf, *DECODE_AS[pf], _ptr(src), w, h, shape[1] * size, _ptr(out), 12 * w]
            fn = lib.fklcase_yuv_to_rgb
        keep = [src]
    else:
        src, out = pixels(h, w, 3), output(h, w, 3)
        a, z = math.radians(case["angle"]), case["zoom"]
        c, s = math.cos(a) / z, math.sin(a) / z
        # about the image's centre
        m = [c, -s, w / 2 - c * w / 2 + s * h / 2, s, c, h / 2 - s * w / 2 - c * h / 2, 0.1 / w, -0.1 / h, 1.0]
        keep = [src, np.array(m, np.float32)]
        args = [stream, _ptr(src), w, h, 3 * w, _ptr(keep[1]), int(case["perspective"]), w, h, _ptr(out), 12 * w]
        fn = lib.fklcase_warp_u8x3
    args = [C.c_int(a) if isinstance(a, int) else a for a in args]
    return functools.partial(fn, *args), out, keep


def run(state):
    for call in state["calls"]:
        if call() != 0:
            raise RuntimeError("the chain was not launched")
    return state["outs"]


def work(case):
    return {k: v * case.get("frames", 1) for k, v in _work_per_frame(case).items()}


def _work_per_frame(case):
    """Bytes of every source pixel the chain looks at and every output, once; arithmetic of the chain per output pixel."""
    kind, w, h = case["kind"], case["w"], case["h"]
    if kind == "thumbs" or kind == "crops":
        n = 5 if kind == "thumbs" else case["batch"]
        px = n * case["dw"] * case["dh"]
        side = [(min(case["lo"], d) + min(case["hi"], d)) / 2 for d in (w, h)]
        # crops overlap: the expected union of n rectangles of the mean size thrown at the image, at most four taps per pixel
        union = w * h * (1.0 - math.exp(-n * side[0] * side[1] / (w * h)))
        return {"bytes": 3 * min(union, 4.0 * px) + px * (3 if kind == "thumbs" else 12), "flops": px * 31.0}
    if kind == "chain":
        return {"bytes": 8.0 * w * h, "flops": float(case["n"]) * w * h}
    if kind == "images":
        return {"bytes": 6.0 * w * h * case["batch"], "flops": 6.0 * w * h * case["batch"]}
    if kind == "nv12":
        px = case["dw"] * case["dh"]
        return {"bytes": min(1.5 * w * h, 12.0 * px) + 12.0 * px, "flops": px * (4 * 18 + 28.0)}
    if kind == "encode" or kind == "decode":
        rows, samples = _frame_shape(case["pf"], w, h)
        size = 2 if case["pf"] == P010 else 1
        return {"bytes": float(rows * samples * size + w * h * 3 * (size if kind == "encode" else 4)), "flops": 18.0 * w * h}
    # the share of the source that an output of the same extent covers is at most all of it
    return {"bytes": 15.0 * w * h, "flops": 40.0 * w * h}


def tolerance(case):
    return "exact"
