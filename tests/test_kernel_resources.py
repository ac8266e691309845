# SPDX-License-Identifier: MPL-2.0
"""Registers of the kernels whose launches count on two workgroups per CU, as the compiler reports them (no GPU)."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_prefill_gemm_leaves_room_for_two_waves_per_simd(tmp_path):
    """The engine's prefill GEMM (a workgroup is one wave per SIMD) in every form but the 64 x 64 residual one over
    Q8_0: two waves per SIMD at least, and nothing spilled in any."""
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                        "-packed-fp32-ops", "-I", os.path.join(ROOT, "include"), "-Rpass-analysis=kernel-resource-usage",
                        "--offload-device-only", "-c", os.path.join(ROOT, "bare.metal_amd", "csrc", "pf_gemm.hip"), "-o",
                        str(tmp_path / "pf_gemm.o")], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
    forms = {}
    for part in r.stderr.split("Function Name: ")[1:]:
        m = re.match(r"\S*k_pf_gemmILi(\d)ELi(\d)ELi(\d)ELi(\d)E", part)
        if m:
            forms[tuple(map(int, m.groups()))] = (int(re.search(r"Occupancy \[waves/SIMD\]: (\d+)", part).group(1)),
                                                  int(re.search(r"VGPRs Spill: (\d+)", part).group(1)))
    assert len(forms) == 20  # formats x (store, swiglu, qkv) x 2 row tiles, residual x 4
    assert {f for f, (waves, spill) in forms.items() if waves < 2} <= {(0, 1, 2, 2)}, forms
    assert {f for f, (waves, spill) in forms.items() if spill} == set(), forms
