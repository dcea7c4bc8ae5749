"""The scalar-base LDS copies (lds_dma16_s, dsa_common.h) hold the wait states
the ISA asks for: 5 between a vector instruction that writes a scalar register
and the vector memory instruction that reads it.  The compiler does not insert
them inside inline asm, so a probe kernel is compiled whose base comes out of
vector registers and its assembly is read."""

from __future__ import annotations

import re
import subprocess

import pytest

from deberta_amd import _build

_PROBE = """
#include "dsa_common.h"
extern "C" __global__ void probe(const char* const* bases, float* out) {
  __shared__ __align__(16) float lds[256];
  const char* base = bases[threadIdx.x >> 6];  // one per wave, held in vector registers
  dsa::%s(base, 16 * (threadIdx.x & 63), lds);
  dsa::vm_wait<0>();
  out[threadIdx.x] = lds[threadIdx.x];
}
"""


@pytest.mark.parametrize("copy", ["lds_dma16_s", "lds_dma16_s_nt"])
def test_scalar_base_waits(copy, tmp_path):
    src, out = tmp_path / "probe.hip", tmp_path / "probe.s"
    src.write_text(_PROBE % copy)
    subprocess.run(
        [_build.hipcc_path(), *_build.HIPCC_FLAGS, "-S", "--offload-device-only", f"-I{_build.CSRC_DIR}", str(src),
         "-o", str(out)],
        check=True, capture_output=True,
    )
    code = [ln.split(";")[0].strip() for ln in out.read_text().splitlines()]
    code = [ln for ln in code if ln and not ln.startswith((".", "#")) and not ln.endswith(":")]
    at = next(n for n, ln in enumerate(code) if ln.startswith("global_load_lds_dwordx4"))
    lo, hi = map(int, re.search(r"s\[(\d+):(\d+)\]", code[at]).groups())
    seen = []
    for reg in range(lo, hi + 1):
        write = max(n for n in range(at) if re.match(rf"v_readfirstlane_b32 s{reg},", code[n]))
        between = code[write + 1:at]
        seen.append(sum(int(ln.split()[1], 0) + 1 if ln.startswith("s_nop") else 1 for ln in between))
    assert min(seen) >= 5, (seen, code[max(0, at - 8):at + 1])
