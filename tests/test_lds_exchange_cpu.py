"""Results on their way out through LDS: what one lane reads another lane of its wave wrote (compiled for the device, nothing is launched)."""
import re
import subprocess

import pytest

import capi

SOURCE = '''#include "kernels/gemm_flex.h"
using namespace paras;
__global__ void probe(const flex::float4v* in, std::uint16_t* dst, long ld, long rows, long cols) {
    __shared__ std::uint16_t stage[4096];
    flex::lds_u16* const out = (flex::lds_u16*)stage;
    const int lane = threadIdx.x & 63;
    flex::RowsOut<2>::lay(out, lane & 15, 0, lane >> 4, flex::pack4<bf16_t>(in[lane]));
    flex::RowsOut<2>::lay(out, lane & 15, 1, lane >> 4, flex::pack4<bf16_t>(in[lane + 64]));
    flex::store_rows<bf16_t, 1, 2>(out, dst, ld, rows, cols, true, false);
}
'''


@pytest.fixture(scope="module")
def steps(tmp_path_factory):
    """LDS accesses and fences of the optimised device code, in its order."""
    where = tmp_path_factory.mktemp("lds")
    (where / "probe.hip").write_text(SOURCE)
    subprocess.run(["/opt/rocm/bin/hipcc", "-O3", "--offload-arch=gfx950", "-std=c++17", "--cuda-device-only", "-S", "-emit-llvm", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                    f"-I{capi.PKG / 'csrc'}", str(where / "probe.hip"), "-o", str(where / "probe.ll")], check=True, capture_output=True)
    body = re.search(r"define [^\n]*probe.*?\n}", (where / "probe.ll").read_text(), re.S)[0]
    kinds = [("write", r"store .*addrspace\(3\)"), ("read", r"load .*addrspace\(3\)"), ("fence", r"fence syncscope\(\"wavefront\"\) (release|acquire)")]
    return [next(k for k, p in kinds if re.search(p, line)) for line in body.splitlines() if any(re.search(p, line) for _, p in kinds)]


def test_the_compiler_may_not_read_rows_before_they_are_laid(steps):
    """Hardware keeps a wave's LDS accesses in order; a compiler that sees a lane's own addresses differ need not."""
    assert steps.count("write") >= 2 and steps.count("read") >= 1
    last, first = max(i for i, s in enumerate(steps) if s == "write"), steps.index("read")
    assert last < first and "fence" in steps[last:first], steps
