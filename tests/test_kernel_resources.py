"""What kernels need when they are compiled for gfx950 (here, without a GPU): no chain makes a kernel that needs scratch memory."""
import os
import re
import subprocess

import pytest

from fusedkernellibrary_amd import build

CSRC = build.CSRC
pytestmark = pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="no hipcc")


def usage(tmp_path, chain, text):
    """{kernel: {resource: number}} of the kernels that `text` makes of a chain."""
    src = tmp_path / "kernels.hip"
    src.write_text(f'#include <hip/hip_runtime.h>\n#define FKD_DEVICE_CODE 1\n#include "{CSRC}/fkd_kernels.hpp"\nusing namespace fkd;\nusing JitChain = {chain};\n{text}\n')
    r = subprocess.run([build.HIPCC, *[f for f in build.HIP_FLAGS if f != "-fPIC"], "--offload-device-only", "-Rpass-analysis=kernel-resource-usage", "-I",
                        build.INCLUDE, "-c", str(src), "-o", str(tmp_path / "kernels.co")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    out = {}
    for name, value in re.findall(r"remark: .*?(Function Name|VGPRs|ScratchSize \[bytes/lane\]|Occupancy \[waves/SIMD\]|LDS Size \[bytes/block\]): (\S+)", r.stderr):
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
