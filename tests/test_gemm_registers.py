"""Spilled registers of the GEMM kernels, from the compiler's own report: a
variant that spills more than the one or two that were measured to be free is
slower than the variant it replaces."""
import os
import re
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "system-lab_amd"))

from smoe import build  # noqa: E402


@pytest.mark.parametrize("name,most", [
    ("smoe_gemm", 1), ("smoe_gemm_packed", 0), ("smoe_gemm_e8m0", 1), ("smoe_gemm_small", 2), ("smoe_gemm_wgrad", 0)])
def test_spilled_registers(name, most):
    src = os.path.join(ROOT, "system-lab_amd", "csrc", name + ".hip")
    flags = [f for f in build.HIP_FLAGS if not f.startswith("-W")]
    r = subprocess.run([build.HIPCC, *flags, "--cuda-device-only", "-Rpass-analysis=kernel-resource-usage", "-c", src,
                        "-o", os.devnull], check=True, capture_output=True, text=True, timeout=600)
    names = re.findall(r"Function Name: (\S+)", r.stderr)
    spills = [int(n) for n in re.findall(r"VGPRs Spill: (\d+)", r.stderr)]
    assert len(names) == len(spills) > 0
    assert max(spills) <= most, [(n, s) for n, s in zip(names, spills) if s > most]
