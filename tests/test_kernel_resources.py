"""Registers of the matrix-core quadrature kernel as the compiler reports them: at the
waves per SIMD it asks for, no form of it spills."""
import os
import re
import subprocess

import pytest

from champ_amd import build


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="needs hipcc")
def test_quadrature_kernel_does_not_spill(tmp_path):
    src = "engine_nonloc.hip"
    r = subprocess.run([build.HIPCC, *build.FLAGS, *build.SOURCE_FLAGS.get(src, []), "--cuda-device-only",
                        "-Rpass-analysis=kernel-resource-usage", "-c", os.path.join(build.CSRC, src), "-o",
                        str(tmp_path / "nonloc.o")], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
    forms = {}
    for part in r.stderr.split("Function Name: ")[1:]:
        if "k_nonloc_mma" in part.split()[0]:
            forms[part.split()[0]] = {k: int(re.search(k + r"[^:]*: (\d+)", part).group(1))
                                      for k in ("VGPRs Spill", "ScratchSize", "Occupancy")}
    assert len(forms) == 8  # orders 2 to 5 in FP64 and FP32
    for name, use in forms.items():
        assert use["VGPRs Spill"] == 0 and use["ScratchSize"] == 0 and use["Occupancy"] >= 3, (name, use)
