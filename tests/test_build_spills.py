"""The build's check that the resident solver's kernels spill no vector registers:
it sees a kernel that does, and takes the compiler's other output as it is."""
import subprocess

import pytest

from tealeaf_opencl_amd import build

# as many live values as `n`, under a bound that leaves a thread 64 registers
SOURCE = """
#include <hip/hip_runtime.h>
template <int N>
__global__ void __launch_bounds__(1024, 8) k_live(double *p)
{
    double v[N];
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = p[i * 1024 + threadIdx.x];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; ++i) p[i * 1024 + threadIdx.x] = v[i] * v[N - 1 - i];
}
template __global__ void k_live<4>(double *);
template __global__ void k_live<64>(double *);
"""


def test_spilling_kernel_is_seen(tmp_path):
    src = tmp_path / "live.hip"
    src.write_text(SOURCE)
    out = subprocess.run(["hipcc", "--offload-arch=" + build.ARCH, "-x", "hip"] + build.COMMON + build.DEVICE_FLAGS +
                         build.USAGE + ["-c", str(src), "-o", str(tmp_path / "live.o")], stdout=subprocess.PIPE,
                         stderr=subprocess.STDOUT, text=True, check=True).stdout
    kernels, spilling = build.spilling_kernels(out)
    assert kernels == 2
    assert len(spilling) == 1 and "ILi64E" in spilling[0]
    assert "remark" not in build._messages(out)


def test_build_refuses_it(tmp_path, monkeypatch):
    (tmp_path / "live.hip").write_text(SOURCE)
    for name, value in (("CSRC", str(tmp_path)), ("LIBDIR", str(tmp_path / "lib")), ("SOURCES", ["live.hip"])):
        monkeypatch.setattr(build, name, value)
    build.build()
    monkeypatch.setattr(build, "NO_SPILL", ("live.hip",))
    with pytest.raises(RuntimeError, match="spill vector registers.*ILi64E.* of 2"):
        build.build()


def test_resident_sources_are_checked():
    assert set(build.NO_SPILL) <= set(build.SOURCES)
