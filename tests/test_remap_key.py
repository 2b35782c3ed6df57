"""Host check of the region-remap threshold key (c-saw_amd/csrc/remap.hpp)
against the search over the normalised CDF it replaces (heur_normalize,
functions.cuh:743-868)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROCM_INC = "/opt/rocm/include"


@pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir(ROCM_INC), reason="needs g++ and HIP headers")
def test_remap_key_matches_normalised_search(tmp_path):
    exe = str(tmp_path / "remap_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM_INC}", "-x", "c++",
                    os.path.join(HERE, "native", "remap_check.cpp"), "-o", exe], check=True, capture_output=True,
                   timeout=240)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=240)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "mismatches=0" in r.stdout
