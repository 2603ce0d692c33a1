"""The fp16 column-batch kernels load rows of B straight into LDS and read them
back transposed.  The wait between the two is written out in the source: the
compiler's own depends on its alias analysis, which a second LDS object in the
kernel misleads.  Checked in the assembly that the source compiles to: every run
of transposed reads of a kernel with such loads follows an explicit wait in its
basic block.
"""
from __future__ import annotations

import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_transposed_reads_follow_an_explicit_wait(tmp_path):
    csrc = os.path.join(ROOT, "xspmm_amd", "csrc")
    out = str(tmp_path / "spmm.s")
    subprocess.run([HIPCC, "-std=c++20", "-O3", "-fPIC", "-I" + os.path.join(ROOT, "include"), "-I" + csrc,
                    "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                    "-S", "--cuda-device-only", os.path.join(csrc, "spmm.hip"), "-o", out],
                   check=True, capture_output=True)
    with open(out) as f:
        text = f.read()
    kernels = 0
    for m in re.finditer(r"^(_ZN\S*spmm_f16_batch_kernel\S*):.*?^\.Lfunc_end", text, re.S | re.M):
        body = m.group(0)
        if " lds\n" not in body:
            continue  # B through registers
        kernels += 1
        runs, waited, reading, asm = 0, None, False, False
        for line in map(str.strip, body.splitlines()):
            if line.startswith(".LBB"):
                waited, reading = None, False
            elif line.startswith((";;#ASMSTART", ";;#ASMEND")):
                asm = line.startswith(";;#ASMSTART")
            elif asm and (w := re.match(r"s_waitcnt vmcnt\((\d+)\)", line)):
                waited = int(w.group(1))
            elif line.startswith("buffer_load"):
                waited, reading = None, False
            elif line.startswith("ds_read_b64_tr") and not reading:
                runs += 1
                reading = True
                # two loads at most were issued after the tile's
                assert waited is not None and waited <= 2, (m.group(1), line)
        assert runs >= 7, m.group(1)  # five pairs of a pass, the last batches
    assert kernels >= 8  # both index types: 128 and 256 columns, by XCD, padded B
