"""Rows brought to LDS by DMA are waited for by the wave that asked for them
before the barrier that hands them to the others: read off the gfx950 assembly,
since a missing wait rarely shows in results.  (CPU: cross-compiled.)"""

import glob
import os
import re
import shlex
import shutil
import subprocess

import pytest

CSRC = glob.glob(os.path.join(os.path.dirname(__file__), "..", "mask-routed*", "csrc"))[0]
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def device_assembly(source, out):
    """Assembly of one source under the Makefile's own flags."""
    dry = subprocess.run(["make", "-n", "-B", f"_build/{source}.o"], cwd=CSRC, check=True,
                         capture_output=True, text=True).stdout
    cmd = next(line for line in dry.splitlines() if f"-c {source}.hip" in line)
    cmd = shlex.split(cmd.split(" -c ")[0])
    subprocess.run(cmd + ["-S", "--cuda-device-only", f"{source}.hip", "-o", str(out)],
                   cwd=CSRC, check=True)
    return out.read_text()


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_routed_dkv_rounds_wait_for_their_rows_before_the_barrier(tmp_path):
    text = device_assembly("routed_attention_bwd", tmp_path / "bwd.s")
    kernels = re.findall(r"^(_ZN\S*routed_attn_dkv_kernelILb([01])ELb([01])E\S*):(.*?)^\.Lfunc_end",
                         text, re.S | re.M)
    assert len(kernels) == 4  # ALiBi x token keep
    for name, _, keep, body in kernels:
        # one round loop per pass: plain and stabilised, or (keep rows) stabilised alone
        passes = 1 if keep == "1" else 2
        joint = re.findall(r"s_waitcnt vmcnt\(0\) lgkmcnt\(0\)\n\s*s_barrier\n\s*;;#ASMEND", body)
        assert len(joint) == passes, name
