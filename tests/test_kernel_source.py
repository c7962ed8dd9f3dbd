"""What the kernels' inline assembly must hold, read from the sources and from their compiled form."""

from __future__ import annotations

import re
import subprocess

from tests.conftest import REPO

CSRC = REPO / "faster-cosyvoice_amd" / "csrc"

PROBE = """
#include "common.hpp"
__global__ void probe(const void* src, float* dst, int n) {
  __shared__ __attribute__((aligned(16))) char smem[4096];
  const uint32_t lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)smem;
  for (int i = 0; i < n; ++i)
    for (int j = 0; j < 4; ++j) fcv::lds_dma16(src, threadIdx.x * 16 + j * 1024, lds + j * 1024);
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  dst[threadIdx.x] = smem[threadIdx.x];
}
"""


def _m0_hazards(asm: str) -> int:
    """LDS copies that directly follow a scalar write of m0."""
    ops = [ln.split(";")[0].strip() for ln in asm.splitlines()]
    ops = [o for o in ops if o and not o.startswith((".", "#")) and not o.endswith(":")]
    return sum(bool(re.match(r"s_\w+ m0,", a)) and "_lds_" in b for a, b in zip(ops, ops[1:]))


def test_lds_copy_waits_for_m0(fcv, tmp_path):
    """gfx9 needs a wait state between a scalar write of m0 and the LDS copy that reads it, which
    nothing inserts inside an inline asm: without it a copy can go to the previous one's address."""
    from faster_cosyvoice_amd import build
    (tmp_path / "probe.hip").write_text(PROBE)
    subprocess.run([build.hipcc(), f"--offload-arch={build.ARCH}", "-O3", "--cuda-device-only", "-S",
                    f"-I{CSRC}", str(tmp_path / "probe.hip"), "-o", str(tmp_path / "probe.s")],
                   check=True, capture_output=True)
    asm = (tmp_path / "probe.s").read_text()
    assert len(re.findall(r"global_load_lds_dwordx4", asm)) >= 4
    assert _m0_hazards(asm) == 0
    # the helper is the only place that writes m0
    writers = [p.name for p in CSRC.iterdir() if re.search(r'"[^"]*\bm0, ', p.read_text())]
    assert writers == ["common.hpp"], writers
