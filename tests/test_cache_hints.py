"""The decoders' two ways to read packed words, as compiled for gfx950: past the
caches (every packed-word load carries the non-temporal bit) and through them
(none does).  With both in one source file the compiler may merge loads that
differ in the hint only, and a merged load has none."""
import pathlib
import re
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

SOURCE = r"""
#include "fls_columns.hpp"
using namespace fls;
template <bool CACHED>
__device__ void decode(const ColDev& c, uint32_t* out) {
    uint32_t x[32];
    decode_regs<false, CACHED>(c, blockIdx.x * 8u + (threadIdx.x >> 5), x);
    for (int r = 0; r < 32; ++r) out[1024u * blockIdx.x + 32 * r + dev::lane32()] = x[r];
}
extern "C" __global__ void decode_cached(const ColDev c, uint32_t* out) { decode<true>(c, out); }
extern "C" __global__ void decode_past(const ColDev c, uint32_t* out) { decode<false>(c, out); }
"""


def loads_of(asm):
    """kernel -> (global loads, those with the non-temporal bit)"""
    found, kernel = {}, None
    for line in asm.splitlines():
        m = re.match(r"^(\w+):", line)
        if m:
            kernel = m.group(1)
        elif re.match(r"\s+(global|flat)_load_dword\s", line):
            n, nt = found.get(kernel, (0, 0))
            found[kernel] = (n + 1, nt + (" nt" in line))
    return found


@pytest.mark.skipif(not pathlib.Path(HIPCC).exists(), reason="no HIP compiler")
def test_packed_words_are_read_as_asked(tmp_path):
    src, asm = tmp_path / "hints.hip", tmp_path / "hints.s"
    src.write_text(SOURCE)
    subprocess.run([HIPCC, "-O3", "-std=c++17", "--offload-arch=gfx950", f"-I{ROOT / 'include'}",
                    f"-I{ROOT / 'fastlanesgpu_amd' / 'csrc'}", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "--cuda-device-only", "-S", str(src), "-o", str(asm)], check=True)
    found = loads_of(asm.read_text())
    words = sum(range(1, 33))  # a load for every packed word of every width
    n, nt = found["decode_cached"]
    assert n >= words and nt == 0, found
    n, nt = found["decode_past"]
    assert nt == words, found
