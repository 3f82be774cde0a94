"""The build's check of the compiler's resource remarks: a kernel compiled for a
stated occupancy must not spill vector registers."""
from aperture3_amd import build

REMARKS = """\
a.hip:5:1: remark: Function Name: {name} [-Rpass-analysis=kernel-resource-usage]
a.hip:5:1: remark:     TotalSGPRs: 106 [-Rpass-analysis=kernel-resource-usage]
a.hip:5:1: remark:     VGPRs: 128 [-Rpass-analysis=kernel-resource-usage]
a.hip:5:1: remark:     SGPRs Spill: 58 [-Rpass-analysis=kernel-resource-usage]
a.hip:5:1: remark:     VGPRs Spill: {spill} [-Rpass-analysis=kernel-resource-usage]
"""
PUSH = "_ZN3apt13k_logsph_pushIdLb1EEEv"


def test_spills_are_found():
    text = (REMARKS.format(name=PUSH, spill=2) + REMARKS.format(name=PUSH, spill=0) +
            REMARKS.format(name="_ZN3apt10k_b_injectIdEEv", spill=464))
    assert build.spilling_kernels(text) == [f"{PUSH}: 2 spills"]


def test_the_compiler_prints_what_is_looked_for(tmp_path):
    """A kernel that cannot keep 200 values in the 64 registers it asks for."""
    src = tmp_path / "spill.hip"
    src.write_text("""#include <hip/hip_runtime.h>
__attribute__((amdgpu_waves_per_eu(8))) __global__ void __launch_bounds__(256)
    k_logsph_push(const double *a, double *b, int n) {
  double v[100];
#pragma unroll
  for (int i = 0; i < 100; i++) v[i] = a[threadIdx.x + i * n];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 100; i++) b[threadIdx.x + (99 - i) * n] = v[i] * v[(i * 7) % 100];
}
""")
    cmd = [build._hipcc(), *build.HIPCC_FLAGS, *build.RESOURCE_REMARKS, "-c", str(src), "-o",
           str(tmp_path / "spill.o")]
    try:
        build._run(cmd)
    except RuntimeError as e:
        assert "k_logsph_push" in str(e) and "spills" in str(e)
    else:
        raise AssertionError("a spilling kernel was accepted")
