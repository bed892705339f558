"""Each kernel that is launched with more than 64 KB of dynamic LDS has had its own limit raised in front. No GPU: a program calls
the library's launch functions with the runtime's calls replaced by ones that keep a record."""
import os
import subprocess

import pytest

SOURCE = r"""
#include <cstdio>
#include <map>
#include "w4a32_layered.h"
#include "w4a32_layered_kernels.h"

static std::map<const void*, size_t> limit;
static int launches, wide, refused;
extern "C" {
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipFuncSetAttribute(const void* f, hipFuncAttribute, int v) { limit[f] = v; return hipSuccess; }
static size_t pushed;
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t lds, hipStream_t) { pushed = lds; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3*, dim3*, size_t* lds, hipStream_t*) { *lds = pushed; return hipSuccess; }
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void**, size_t lds, hipStream_t) {
  ++launches;
  if (lds > 64 * 1024) {
    ++wide;
    const auto it = limit.find(f);
    if (it == limit.end() || it->second < lds) ++refused;
  }
  return hipSuccess;
}
}

int main() {
  for (int dtype : {W4A32_LAYERED_BF16, W4A32_LAYERED_F32})
    for (int experts : {1, 16, 1, 80}) {  // the router inside the experts' launch, in front, inside, in front
      w4::MoeGeom g{16448, 16448, 24, 64, experts, 1, 7.0f};
      w4::RowPrologue pro{};
      if (w4::launch_moe_decode(dtype, g, pro, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr) != hipSuccess)
        return 2;
      if (w4::moe_routes_itself(dtype == W4A32_LAYERED_BF16 ? 2 : 4, g) != (experts == 1)) return 3;
    }
  printf("%d launches, %d wide, %d refused\n", launches, wide, refused);
}
"""


def test_experts_of_a_wide_decode_step(pkg, tmp_path):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    here = os.path.dirname(pkg.__file__)
    src, exe = tmp_path / "lds.hip", tmp_path / "lds"
    src.write_text(SOURCE)
    pkg.lib()
    subprocess.run([hipcc, "--offload-arch=gfx950", "-O1", "-std=c++17", "-rdynamic", f"-I{here}/csrc", f"-I{here}/../include", str(src), "-o",
                    str(exe), f"-L{here}", "-lw4a32_hip", f"-Wl,-rpath,{here}"], check=True, capture_output=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert (out.returncode, out.stdout) == (0, "16 launches, 8 wide, 0 refused\n")
