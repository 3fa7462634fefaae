"""The grid rules of the kernels that split groups of rates or time steps over
blockIdx.y (csrc/rate_groups.h), on the host: a part without a group would index
before the kernels' tables, and a wrapped product would leave groups out."""
import shutil
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).parent
CSRC = HERE.parent / "frequencydriftratetransforms.jl_amd" / "csrc"


def test_parts_take_every_group_once(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no g++")
    exe = tmp_path / "rate_groups"
    subprocess.run([gxx, "-O1", "-std=c++17", "-Wall", f"-I{CSRC}", str(HERE / "rate_groups.cpp"), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
