"""The build refuses kernels that count their loads in flight themselves where the compiler puts some of their registers into memory."""
import glob
import os
import re

import pytest

from flexllm_amd import build

# 300 values that live across a barrier where a thread has 64 registers
SOURCE = """#include <hip/hip_runtime.h>
__global__ __launch_bounds__(1024, 8) void NAME(const float* x, float* y) {
    float v[300];
    for (int i = 0; i < 300; i++) v[i] = x[i * 1024 + threadIdx.x];
    __syncthreads();
    for (int i = 0; i < 300; i++) y[i * 1024 + threadIdx.x] = v[i] * v[299 - i];
}
"""


@pytest.mark.parametrize("name,refused", [("gemm_few_kernel", True), ("walk_kernel", True), ("some_kernel", False)])
def test_spills(tmp_path, name, refused):
    src = tmp_path / "k.hip"
    src.write_text(SOURCE.replace("NAME", name).replace("for (int i", "_Pragma(\"unroll\") for (int i"))
    run = lambda: build.build(srcs=[str(src)], out=str(tmp_path / "k.so"), obj_dir=str(tmp_path))  # noqa: E731
    if refused:
        with pytest.raises(RuntimeError, match=name):
            run()
    else:
        assert os.path.exists(run())


def test_names_are_kernels():
    text = "".join(open(f).read() for f in glob.glob(os.path.join(build.CSRC, "*")) if f.endswith((".h", ".hip")))
    for name in build.WITHOUT_SPILLS:
        assert re.search(r"__global__[^;{]*\b%s\(" % name, text), name


def test_what_is_no_remark_is_kept():
    out = """In file included from a.hip:1:
a.h:3:1: warning: something [-Wsomething]
    3 | int x;
      | ^
In file included from a.hip:1:
./a.h:9:1: remark: Function Name: gemm_few_kernel [-Rpass-analysis=kernel-resource-usage]
    9 | void gemm_few_kernel() {
      | ^
./a.h:9:1: remark:     ScratchSize [bytes/lane]: 16 [-Rpass-analysis=kernel-resource-usage]
./a.h:9:1: remark:     VGPRs Spill: 4 [-Rpass-analysis=kernel-resource-usage]
'-packed-fp32-ops' is not a recognized feature for this target (ignoring feature)
a.hip:9:1: error: other"""
    kernels, rest = build.resources(out)
    assert kernels == {"gemm_few_kernel": {"ScratchSize": 16, "VGPRs Spill": 4}} and build.spilled(kernels) == ["gemm_few_kernel"]
    assert rest == out.splitlines()[:4] + ["a.hip:9:1: error: other"]


def test_the_compiler_knows_who_writes_m0():
    """m0 has the LDS address of a direct load: a statement that writes it puts back what was there, or names it among its operands."""
    for f in glob.glob(os.path.join(build.CSRC, "*")):
        if f.endswith((".h", ".hip")):
            for asm in re.findall(r"\basm volatile\((.*?)\);", open(f).read(), re.S):
                if "global_load_lds" in asm or re.search(r"\bm0\b", asm):
                    assert "{m0}" in asm or ("s_mov_b32 %0, m0" in asm and "s_mov_b32 m0, %0" in asm), (f, asm)
