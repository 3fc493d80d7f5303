"""The coarse tail's levels lie inside the LDS that its launches ask for (csrc/wl_tail.h, compiled on
the CPU): the image's rounding up to whole vectors is part of the request, for the single flow's launch
and for the batch's, which takes the largest member's."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "waterlily.jl_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_every_tail_array_lies_in_the_requested_lds(tmp_path):
    exe = str(tmp_path / "tail_layout")
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, "-o", exe, os.path.join(HERE, "c", "tail_layout.cpp")],
                   check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True, timeout=120)
    bad, rest = out.stdout.strip().split(" of ")
    assert bad == "0" and rest.endswith("some padded"), out.stdout
