"""Vector loads at addresses that need not be multiples of their size must not promise the compiler that they are: the sources with such
loads compile without -Walign-mismatch, and the library is built with it as an error."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cutile.jl_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_layernorm_rows_of_any_alignment():
    run = subprocess.run([HIPCC, "--offload-arch=gfx950", "--cuda-device-only", "-std=c++17", "-fsyntax-only", "-Werror=align-mismatch", "layernorm.hip"],
                         cwd=CSRC, capture_output=True, text=True)
    assert run.returncode == 0, run.stderr


def test_the_build_refuses_such_loads():
    with open(os.path.join(CSRC, "Makefile")) as f:
        assert "-Werror=align-mismatch" in f.read()
