"""The projection GEMM's K loop in gfx950 assembly: the LDS reads of a stage's operands all
come before the barrier after which the other waves' direct loads overwrite that stage.

A wave reads k steps 1 to 3 of a stage (2 W and MT / 64 x operands each) in the block that ends
in the stage barrier; step 0 was read behind the barrier before it."""
import os
import re
import subprocess
import tempfile

import pytest

from prefixlm import _build

CSRC = _build.CSRC
SOURCE = """#include <hip/hip_runtime.h>
#include "gemm.h"
using namespace prefixlm;
template __global__ void mlp::proj_gemm_kernel<256, false, true>(mlp::Params);
template __global__ void mlp::proj_gemm_kernel<256, true, true>(mlp::Params);
template __global__ void mlp::proj_gemm_kernel<256, true, false>(mlp::Params);
template __global__ void mlp::proj_gemm_kernel<256, false, false>(mlp::Params);
template __global__ void mlp::proj_gemm_kernel<128, false, true>(mlp::Params);
template __global__ void mlp::proj_gemm_kernel<128, true, true>(mlp::Params);
template __global__ void mlp::proj_gemm_kernel<128, true, false>(mlp::Params);
template __global__ void mlp::proj_gemm_kernel<128, false, false>(mlp::Params);
"""


def _kernels():
    try:
        hipcc = _build.hipcc()
    except RuntimeError:
        pytest.skip("hipcc not found")
    flags = [f for f in _build.HIP_FLAGS if f not in ("-fPIC", "-shared")]
    with tempfile.TemporaryDirectory() as d:
        src, asm = os.path.join(d, "k.hip"), os.path.join(d, "k.s")
        with open(src, "w") as f:
            f.write(SOURCE)
        subprocess.run([hipcc, *flags, f"-I{CSRC}", "--cuda-device-only", "-S", src, "-o", asm], check=True,
                       capture_output=True)
        with open(asm) as f:
            text = f.read()
    return re.findall(r"^_ZN8prefixlm3mlp16proj_gemm_kernelILi(\d+)(\w+):.*?\n(.*?)^\.Lfunc_end", text, re.M | re.S)


def test_stage_reads_end_before_the_barrier():
    kernels = _kernels()
    assert len(kernels) == 8
    for mt, name, body in kernels:
        blocks = re.split(r"^\.LBB\w+:.*$", body, flags=re.M)
        loop = [b for b in blocks if "s_barrier" in b and "v_mfma" in b]
        assert len(loop) == 1, (mt, name)
        before = loop[0].split("s_barrier")[0]
        assert before.count("ds_read_b128") == 3 * (2 + int(mt) // 64), (mt, name)
