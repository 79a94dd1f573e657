"""Numbers that lanes of a wave pass to each other through LDS (partial row sums, the row patches of the stores) are written and read
on the two sides of a fence.  The compiled form of the helpers is looked at: one kernel per helper, as LLVM IR."""
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "kernels_amd", "csrc")
HIPCC = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")
SOURCE = """
#include <hip/hip_runtime.h>
#include "sa_common.h"
#include "sa_fwd.h"
#include "sa_bwd.h"
#include "sa_f32.h"
using namespace sa;
extern __shared__ __attribute__((aligned(16))) char lds[];
extern "C" __global__ void dots_16(const __bf16* o, float* out) {
  RowDots<__bf16, 64> d;
  d.load(o, 64, 0, 31, threadIdx.x);
  d.partial((const __bf16*)lds, (float*)(lds + 8192), threadIdx.x);
  out[threadIdx.x] = RowDots<__bf16, 64>::total((const float*)(lds + 8192), threadIdx.x);
}
extern "C" __global__ void dots_32(const float* o, float* out) {
  RowDots32<64> d;
  d.load(o, 64, 0, 31, threadIdx.x);
  d.partial((const float*)lds, (float*)(lds + 8192), threadIdx.x);
  out[threadIdx.x] = RowDots32<64>::total((const float*)(lds + 8192), threadIdx.x);
}
extern "C" __global__ void rows_16(const f32x16* in, __bf16* out) {
  f32x16 acc[2] = {in[2 * threadIdx.x], in[2 * threadIdx.x + 1]};
  store_rows_coalesced<__bf16, 64, 2>((__bf16*)lds, out, 32, acc, 1.0f, threadIdx.x);
}
extern "C" __global__ void rows_32(const f32x16* in, float* out) {
  f32x16 acc[4] = {in[4 * threadIdx.x], in[4 * threadIdx.x + 1], in[4 * threadIdx.x + 2], in[4 * threadIdx.x + 3]};
  store_rows_f32<128, false>((float*)lds, out, 32, acc, 1.0f, threadIdx.x);
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no compiler")
def test_writes_and_reads_of_a_wave_are_fenced(tmp_path):
    (tmp_path / "t.hip").write_text(SOURCE)
    subprocess.run([HIPCC, "-O1", "--offload-arch=gfx950", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "--cuda-device-only", "-S", "-emit-llvm", "-I", CSRC,
                    "t.hip", "-o", "t.ll"], cwd=tmp_path, check=True, capture_output=True)
    ir = (tmp_path / "t.ll").read_text()
    for kernel, exchanges in (("dots_16", 1), ("dots_32", 1), ("rows_16", 1), ("rows_32", 2)):
        body = re.search(r"define[^\n]*@%s\(.*?^}" % kernel, ir, re.S | re.M).group(0)
        # 'w'rite or 'r'ead of LDS, '|' the pair of fences around a wave barrier
        events = ""
        for line in body.splitlines():
            if "store " in line and "addrspace(3)" in line:
                events += "w"
            elif "load " in line and "addrspace(3)" in line:
                events += "r"
            elif 'fence syncscope("wavefront")' in line:
                events += "|"
        assert re.search(r"w[|]+r", events), (kernel, events)
        turns = re.sub(r"(.)\1+", r"\1", events)          # without repetitions
        assert turns.count("w|r") == exchanges, (kernel, turns)
        if kernel.startswith("rows"):
            assert "wr" not in turns and "rw" not in turns, (kernel, turns)
