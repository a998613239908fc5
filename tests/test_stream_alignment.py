"""The streaming row load claims no more alignment than the interface promises (no GPU).

Rows of 4-byte texels begin at any multiple of 4 bytes.  A kernel that loads four
texels with loadRowStream is compiled to the compiler's intermediate form, where
every non-temporal load must say 4 bytes, and to instructions, where it must still
be one 16-byte load with the hint.
"""
import os
import re
import shutil
import subprocess

import pytest

from vk_compute_mipmaps_amd import build

SOURCE = """
#include "kernel_common.hpp"
using namespace nvpro_pyramid;
__global__ void streamedRow(const uint8_t* p, uint32_t* out)
{
  Srgba8::Raw t[4];
  loadRowStream<Srgba8, 4>(p + 4u * threadIdx.x, t);
  out[threadIdx.x] = t[0] ^ t[1] ^ t[2] ^ t[3];
}
"""


@pytest.mark.skipif(not (os.path.exists(build.hipcc()) or shutil.which("hipcc")), reason="needs hipcc")
def test_streamed_rows_are_loaded_at_four_byte_alignment(tmp_path):
    source = tmp_path / "streamed_row.hip"
    source.write_text(SOURCE)
    made = {}
    for kind, flags in (("ll", ["-S", "-emit-llvm"]), ("s", ["-S"])):
        out = tmp_path / f"streamed_row.{kind}"
        cmd = [build.hipcc(), *build.HIPCC_FLAGS, "-I", build.INCLUDE, "-I", build.CSRC, "--offload-device-only", *flags,
               str(source), "-o", str(out)]
        run = subprocess.run(cmd, capture_output=True, text=True)
        assert run.returncode == 0, run.stderr[-4000:]
        made[kind] = out.read_text()
    loads = [line for line in made["ll"].splitlines() if " load " in line and "!nontemporal" in line]
    assert loads and all(re.search(r"\balign 4\b", line) for line in loads), loads
    assert len(re.findall(r"global_load_dwordx4 .*\bnt\b", made["s"])) == 1
