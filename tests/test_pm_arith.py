"""Host-side check of the integer path's two-word products (primes just below a
power of two) and of the bounds its butterflies keep from stage to stage."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_two_word_products_and_butterfly_bounds(tmp_path):
    exe = str(tmp_path / "pm_check")
    subprocess.run([HIPCC, "-O2", "-std=c++17", "-x", "hip", "--offload-arch=gfx950",
                    "-I", os.path.join(ROOT, "privacy-rag_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "pm_arith_check.cpp"), "-o", exe],
                   check=True, capture_output=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0 and "ALL OK" in r.stdout, r.stdout
