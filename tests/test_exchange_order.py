"""An exchange through LDS keeps its reads before its closing barrier.

A register-Stockham fastconv branches right after an exchange (on its scale),
and the compiler had sunk the exchange's reads past the closing barrier to their
uses behind that branch: a wave that was late could then read what a faster wave
had already written for the next exchange.  Two barriers with no LDS access
between them are the mark of it, so the test compiles such kernels for gfx950
and looks at the order of the LDS accesses and barriers in their assembly."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

SOURCE = """
#include "ovx_row_dev.hpp"
using namespace ovx;
template <int N, int P>
__global__ __launch_bounds__(N / P) void k(const float2 *x, const float2 *w, float2 *y, long rows, const float2 *tw,
                                           float scale)
{
  __shared__ float2 lds[Engine<N, P>::LROW];
  row_fastconv_body<N, P>(x, N, w, 0, y, N, rows, tw, scale, blockIdx.x, 0, threadIdx.x, lds);
}
template __global__ void k<4096, 16>(const float2 *, const float2 *, float2 *, long, const float2 *, float);
template __global__ void k<3072, 12>(const float2 *, const float2 *, float2 *, long, const float2 *, float);
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_no_exchange_reads_after_its_closing_barrier(tmp_path):
    src, out = tmp_path / "k.hip", tmp_path / "k.s"
    src.write_text(SOURCE)
    subprocess.run([HIPCC, "-O3", "-std=c++17", "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-ffp-contract=fast", "-w", "--cuda-device-only", "-S",
                    "-I" + os.path.join(ROOT, "openvsip_amd", "csrc"), str(src), "-o", str(out)], check=True,
                   stderr=subprocess.DEVNULL)
    bodies = re.split(r"\n(?=_Z\w+:)", out.read_text())
    kernels = [b.split(".section", 1)[0] for b in bodies if b.startswith("_Z")]
    assert len(kernels) == 2
    for body in kernels:
        seen = re.findall(r"^\s+(s_barrier|ds_read|ds_write)", body, re.M)
        assert seen.count("s_barrier") >= 8
        assert not any(a == b == "s_barrier" for a, b in zip(seen, seen[1:]))
