"""What the compiler does not see of the direct-to-LDS loads of csrc/kernels/flash_pipe.h: their wait
states, read off the assembly of a small kernel (hipcc cross-compiles without a GPU)."""
import os
import re
import subprocess

from loqa_hub_amd._native import build

# a base that a v_readlane has just made, as the page lookup does
KERNEL = """
#include "flash_pipe.h"
__global__ void probe(const unsigned long long* pages, int n, float* out) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const unsigned long long at = pages[threadIdx.x];
  const unsigned lo = __builtin_amdgcn_readlane((unsigned)at, n), hi = __builtin_amdgcn_readlane((unsigned)(at >> 32), n);
  fl_load_lds((const bf16_t*)(((unsigned long long)hi << 32) | lo), threadIdx.x * 16, fl_lds_at(lds));
  fl_sync();
  out[threadIdx.x] = ((float*)lds)[threadIdx.x];
}
"""


def test_scalar_base_of_a_load_is_ready(tmp_path):
    src, out = tmp_path / "probe.hip", tmp_path / "probe.s"
    src.write_text(KERNEL)
    subprocess.run([build._hipcc(), "--offload-arch=gfx950", "-O3", "-std=c++17", f"-I{os.path.join(build.CSRC, 'kernels')}",
                    *build.NO_PACKED_F32, "--cuda-device-only", "-S", str(src), "-o", str(out)], check=True, capture_output=True)
    code = [x.strip() for x in out.read_text().splitlines()]
    code = [x for x in code if re.match(r"(s|v|ds|global|buffer|flat)_", x)]
    (at, load), = [(i, x) for i, x in enumerate(code) if x.startswith("global_load_lds_dwordx4")]
    first, last = map(int, re.search(r"s\[(\d+):(\d+)\]", load).groups())
    waited = 0
    for x in reversed(code[:at]):
        to = re.match(r"\S+ s(?:\[(\d+):(\d+)\]|(\d+))", x)
        if to and (int(to[1]) <= last and int(to[2]) >= first if to[1] else first <= int(to[3]) <= last):
            assert x.startswith("s_") or waited >= 5, (x, load, waited)
            break
        waited += int(x.split()[1]) + 1 if x.startswith("s_nop") else 1
    else:
        raise AssertionError("no writer of the base")
