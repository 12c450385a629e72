"""What the kernels' wide memory accesses tell the compiler about their addresses, read from the intermediate code of a small kernel
built with the library's flags: accesses to rows at any byte promise nothing, those at dword boundaries a dword.  (A promise that
does not hold would still run today and leave the optimiser free to break it.)"""
import os
import re
import subprocess

import pytest

from fusedkernellibrary_amd.build import HIP_FLAGS, HIPCC, INCLUDE

PRELUDE = """
#include <hip/hip_runtime.h>
#define FKD_DEVICE_CODE 1
#include "fkd/ops.hpp"
using namespace fkd;
using Px = Vec<u8, 3>;
using F4 = Vec<f32, 4>;
template <int W, bool ALIGNED> __device__ void words(const char* a, char* b) {
    u32 w[W];
    detail::load_words<W, false, ALIGNED>(a, w);
    detail::store_words<W, ALIGNED>(b, w);
}
template <int W, bool ALIGNED> __device__ void streamed(const char* a, char* b) {
    u32 w[W];
    detail::load_words<W, true, ALIGNED>(a, w);
    detail::store_words<W, ALIGNED>(b, w);
}
template <bool ALIGNED> __device__ void exchanged(const char* a, char* b) {
    u32 w[12];
    detail::load_words_wave<12, false, ALIGNED>(a, w);
    detail::store_words_wave<12, ALIGNED>(b, w);
}
template <class T> __device__ void pair_window(const char* a, char* b, u32 off) {
    Vec<f32, 2> sum{};
    T x{}, y{};
    detail::pair_window_values<false, T>(detail::load_pair_window<T>(a, off), x, y);
    sum.x = f32(chan<0>(x)); sum.y = f32(chan<0>(y));
    detail::store_elem_at<Vec<f32, 2>>(b, off, sum);
}
__device__ void shifted_window(const char* a, char* b, u32 off) {
    const auto window = detail::load_pair_window<Px>(a, off);
    detail::store_words<3>(b, window.w);
}
__device__ void runs(const char* a, char* b, u32 off) {
    const auto bits = detail::load_bits_at<F4, 1, false>(a, off);
    Slot<F4> one[1];
    one[0].v = detail::run_value<0>(bits);
    detail::store_run_at<F4, 1>(b, off, one);
}
"""

CASES = [
    *[(f"words<{w}, {aligned}>(a, b)", 4 if aligned == "true" else 1) for w in (1, 2, 3, 4, 8) for aligned in ("true", "false")],
    ("streamed<3, false>(a, b)", 1), ("streamed<4, true>(a, b)", 4), ("exchanged<false>(a, b)", 1), ("exchanged<true>(a, b)", 4),
    ("pair_window<Vec<u8, 4>>(a, b, off)", 1), ("runs(a, b, off)", 1),
    ("shifted_window(a, b, off)", 4)]


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """The intermediate code of one kernel per case."""
    src = tmp_path_factory.mktemp("access") / "probe.hip"
    src.write_text(PRELUDE + "\n".join(f'extern "C" __global__ void probe{i}(const char* a, char* b, u32 off) {{ {body}; }}'
                                       for i, (body, _) in enumerate(CASES)))
    out = src.with_suffix(".ll")
    r = subprocess.run([HIPCC, *HIP_FLAGS, "-I", INCLUDE, "--cuda-device-only", "-emit-llvm", "-S", str(src), "-o", str(out)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    text = out.read_text()
    return [text[text.index(f"@probe{i}("):].split("\n}", 1)[0] for i in range(len(CASES))]


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
@pytest.mark.parametrize("i", range(len(CASES)), ids=[c[0] for c in CASES])
def test_wide_accesses_promise_no_more_than_they_know(kernels, i):
    found = [int(m) for m in re.findall(r"(?:load|store) [^\n]*addrspace\(1\)[^\n]*, align (\d+)", kernels[i])]
    assert found and set(found) == {CASES[i][1]}, kernels[i]
