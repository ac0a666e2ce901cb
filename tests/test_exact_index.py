"""Addresses and routes of the fp32-matrix kernels, walked on the host."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def run_host(name, tmp_path):
    cxx = shutil.which("g++") or shutil.which("clang++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = tmp_path / name
    subprocess.run([cxx, "-std=c++17", "-Wall", "-Werror",
                    "-I", os.path.join(ROOT, "neonengine_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", name + ".cpp"), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[-3000:]


def test_expert_input_addresses_stay_inside_the_row(tmp_path):
    """Rows of 33-47, 65-79 and 97-111 units have 3, 5 or 7 groups of 16 and run
    in the kernels of 4, 6 and 8: the group past the row reads inside it too."""
    run_host("exact_index", tmp_path)


def test_routes_lie_where_they_were_measured(tmp_path):
    """Sizes timed on both sides of each line take the form that was faster."""
    run_host("exact_routes", tmp_path)
