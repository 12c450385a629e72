"""Kernels compiled for gfx950 (here, without a GPU): no chain makes a kernel that needs scratch memory, and a warp requests all its taps before it
waits for one."""
import os
import re
import subprocess

import pytest

from fusedkernellibrary_amd import build

CSRC = build.CSRC
pytestmark = pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="no hipcc")


def compiled(tmp_path, chain, text, *flags):
    """The output (path) and the remarks of compiling `text`, which makes kernels of a chain."""
    src, out = tmp_path / "kernels.hip", tmp_path / "kernels.out"
    src.write_text(f'#include <hip/hip_runtime.h>\n#define FKD_DEVICE_CODE 1\n#include "{CSRC}/fkd_kernels.hpp"\nusing namespace fkd;\nusing JitChain = {chain};\n{text}\n')
    r = subprocess.run([build.HIPCC, *[f for f in build.HIP_FLAGS if f != "-fPIC"], "--offload-device-only", "-I", build.INCLUDE, *flags, str(src), "-o", str(out)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    return out, r.stderr


def usage(tmp_path, chain, text):
    """{kernel: {resource: number}} of the kernels that `text` makes of a chain."""
    remarks = compiled(tmp_path, chain, text, "-c", "-Rpass-analysis=kernel-resource-usage")[1]
    out = {}
    for name, value in re.findall(r"remark: .*?(Function Name|VGPRs|ScratchSize \[bytes/lane\]|Occupancy \[waves/SIMD\]|LDS Size \[bytes/block\]): (\S+)", remarks):
        if name == "Function Name": last = out.setdefault(value, {})
        else: last[name.split(" ")[0]] = int(value)
    return out


def muls(n, t="Vec<f32,4>"):
    return ",".join([f"Mul<{t},{t},{t}>"] * n)


@pytest.mark.parametrize("ops", [8, 9, 60])
def test_long_chains_behind_a_warp_need_no_scratch_memory(tmp_path, ops):
    """More registers than eight waves leave are taken, not spilled: the build refuses kernels that need scratch memory."""
    chain = f"Chain<Warp<1,Read2D<Vec<u8,4>>>,OpList<{muls(ops)}>,Write2D<Vec<f32,4>>>"
    kernels = "\n".join(f"template __global__ void fkd::k_rows<JitChain, 4, 1, false, {form}>(const typename JitChain::Params, const TileGeom);" for form in ("kRowsLines", "kRowsSmall"))
    got = usage(tmp_path, chain, kernels)
    assert len(got) == 2 and all(u["ScratchSize"] == 0 for u in got.values())


@pytest.mark.parametrize("pixel,out", [("f32", "f32"), ("u8", "f32"), ("Vec<u8,3>", "Vec<f32,3>"), ("Vec<u8,4>", "Vec<f32,4>"), ("Vec<u16,3>", "Vec<f32,3>")])
def test_a_warp_waits_for_no_tap_before_it_has_requested_all(tmp_path, pixel, out):
    """Four pixels of two source rows: eight loads of pairs of taps leave before the first wait, in each variant of the kernel."""
    kernels = "\n".join(f"template __global__ void fkd::k_rows<JitChain, 4, 1, false, {form}>(const typename JitChain::Params, const TileGeom);" for form in ("kRowsLines", "kRowsSmall"))
    asm = compiled(tmp_path, f"Chain<Warp<0,Read2D<{pixel}>>,OpList<>,Write2D<{out}>>", kernels, "-S")[0].read_text()
    groups = [0]
    for line in asm.splitlines():
        if re.match(r"\s+buffer_load", line): groups[-1] += 1
        elif re.match(r"\s+s_waitcnt.*vmcnt", line) and groups[-1]: groups.append(0)
    assert [g for g in groups if g] == [8, 8, 8]        # (the kernel for larger outputs has a variant for waves inside the image)
