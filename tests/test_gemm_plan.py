"""How the fp32 GEMMs are cut into workgroups, at extents up to the largest
that the entry points take (CPU: the rules are host code)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_gemm_plans(tmp_path):
    exe = tmp_path / "gemm_plan_check"
    build = subprocess.run(["g++", "-O2", "-std=c++20", f"-I{ROOT / 'rushlite_amd' / 'csrc' / 'hip'}",
                            str(ROOT / "tests" / "native" / "gemm_plan_check.cpp"), "-o", str(exe)],
                           capture_output=True, text=True)
    assert build.returncode == 0, build.stderr
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
    assert "gemm plans ok" in out.stdout
