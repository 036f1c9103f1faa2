"""
Kernels whose launches count on two workgroups per CU: the compiler must leave them the registers for it.  Compiled here, as
the library is, for what the compiler reports; no GPU.
"""
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "heat_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc"


def _resources(source, tmp_path):
    """{kernel: {"waves": per SIMD, "spilled": vector registers}} of one source file with the library's own flags."""
    line = subprocess.run(["make", "-B", "-n", "-C", CSRC, "-s", source.replace(".hip", ".o")], capture_output=True, text=True,
                          check=True).stdout.strip().splitlines()[-1].split()
    line = line[: line.index("-o")] + ["-o", str(tmp_path / "device.o"), "--cuda-device-only",
                                       "-Rpass-analysis=kernel-resource-usage"]
    report = subprocess.run(line, cwd=CSRC, capture_output=True, text=True, check=True).stderr
    out = {}
    for name, body in re.findall(r"Function Name: (\S+)(.*?)(?=Function Name:|\Z)", report, re.S):
        out[name] = {"waves": int(re.search(r"Occupancy \[waves/SIMD\]: (\d+)", body).group(1)),
                     "spilled": int(re.search(r"VGPRs Spill: (\d+)", body).group(1))}
    return out


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs the compiler")
def test_exact_kernels_run_two_workgroups_per_cu(tmp_path):
    kernels = _resources("hkm_assign_wide.hip", tmp_path)
    # workgroups of four waves, one on each SIMD
    for part in ("wide_exact_kernel", "panel_exact_kernel"):
        found = [v for n, v in kernels.items() if part in n]
        assert found, part
        for v in found:
            assert v["waves"] >= 2 and v["spilled"] == 0, (part, v)


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs the compiler")
def test_one_product_kernels_keep_their_registers(tmp_path):
    found = {n: v for n, v in _resources("hkm_assign_wide.hip", tmp_path).items() if "assign_panel_kernel" in n}
    assert len(found) == 6
    for n, v in found.items():
        assert v["waves"] >= 2 and v["spilled"] == 0, (n, v)
