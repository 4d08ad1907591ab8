"""Integer code shared by the host and the kernels, run on the CPU by a driver of
its own (csrc/host_checks.cpp, plain C++)."""
import os
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "maxwellfdm.jl_amd", "csrc")


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("host_checks") / "host_checks")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "host_checks.cpp", "-o", exe], cwd=CSRC, check=True)
    return exe


def run(driver, *args):
    p = subprocess.run([driver, *map(str, args)], capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, p.stdout + p.stderr
    return p.stdout


def test_resident_index(driver):
    """The resident solver's cells, halo, exchange and staging places, for every
    box shape on grids at and around its edges and its limit of boxes, with every
    combination of ends, reflections and component windows: each access inside
    its array, each staged place written once, each exchanged value read where
    its owner writes it."""
    assert "resident ok" in run(driver, "resident")
