"""Registers of kernels whose speed hangs on them, from the compiler's own report for gfx950."""
from __future__ import annotations

import re
import subprocess

from isar_imaging_cuda_amd import build as B


def test_chirp_z_kernels_do_not_spill(tmp_path):
    """Every chirp-z kernel keeps its data in vector registers, at four waves a SIMD: with 14 to 27 of them in
    scratch memory the lengths other than 2 M were up to a fifth slower than a form that waits for each load."""
    src = B.CSRC / "kernels" / "mtrc.hip"
    cmd = [B.HIPCC, *B.HIP_FLAGS, *B.HIP_FILE_FLAGS.get(src.name, []), "-I", str(B.INC), "-I", str(B.CSRC), "-c", str(src),
           "-o", str(tmp_path / "mtrc.o"), "-Rpass-analysis=kernel-resource-usage"]
    report = subprocess.run(cmd, capture_output=True, text=True, check=True).stderr
    spills = dict(re.findall(r"Function Name: (\S+).*?VGPRs Spill: (\d+)", report, re.S))
    chirp_z = {k: int(v) for k, v in spills.items() if "k_mtrc_czt" in k}
    assert len(chirp_z) == 18 and not any(chirp_z.values()), chirp_z
