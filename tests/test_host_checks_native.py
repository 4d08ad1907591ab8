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


# (box, grid, components, vectors, scene, right-hand sides, µs per step resident, step by step), measured
MEASURED = [
    ((8, 4, 4), (16, 16, 16), 3, "fp64", "diag", 1, 7.4, 19.6),
    ((8, 4, 4), (16, 16, 16), 3, "fp64", "diag", 16, 17.5, 27.1),
    ((8, 4, 4), (24, 24, 24), 3, "fp64", "diag", 2, 9.4, 21.6),
    ((8, 4, 4), (24, 24, 24), 3, "fp64", "diag", 16, 70.3, 39.4),
    ((8, 4, 4), (31, 31, 32), 3, "fp64", "diag", 1, 9.4, 22.1),
    ((8, 4, 4), (31, 31, 32), 3, "fp64", "diag", 2, 20.4, 25.1),
    ((8, 4, 4), (31, 31, 32), 3, "fp64", "diag", 4, 39.6, 30.6),
    ((8, 4, 4), (31, 31, 32), 3, "fp64", "diag", 16, 156.8, 60.1),
    ((8, 8, 4), (36, 36, 36), 3, "fp64", "diag", 2, 21.7, 30.6),
    ((8, 8, 4), (36, 36, 36), 3, "fp64", "diag", 6, 63.8, 45.7),
    ((16, 8, 4), (48, 48, 48), 3, "fp64", "diag", 2, 28.1, 39.6),
    ((16, 8, 4), (48, 48, 48), 3, "fp64", "diag", 16, 220.6, 180.4),
    ((16, 8, 4), (48, 48, 48), 3, "fp64", "mu", 2, 30.9, 43.4),
    ((16, 8, 4), (48, 48, 48), 3, "fp64", "mu", 16, 242.6, 216.5),
    ((8, 8, 4), (36, 36, 36), 3, "fp64", "full", 2, 23.1, 39.1),
    ((8, 8, 4), (36, 36, 36), 3, "fp64", "full", 16, 178.9, 124.5),
    ((8, 8, 4), (36, 36, 36), 3, "fp32", "diag", 2, 20.7, 29.6),
    ((8, 8, 4), (36, 36, 36), 3, "fp32", "diag", 16, 159.5, 70.0),
    ((16, 8, 4), (48, 48, 48), 3, "fp32", "diag", 8, 100.4, 70.6),
    ((16, 8, 1), (150, 120, 1), 2, "fp64", "diag", 16, 119.7, 35.0),
    ((16, 8, 1), (150, 120, 1), 3, "fp32", "mu", 1, 7.7, 18.4),
    ((32, 16, 1), (350, 360, 1), 2, "fp64", "full", 1, 11.8, 25.3),
    ((32, 16, 1), (350, 360, 1), 2, "fp64", "full", 16, 199.7, 178.7),
    ((32, 16, 1), (200, 301, 1), 1, "fp32", "diag", 16, 152.1, 40.3),
    ((32, 32, 1), (500, 500, 1), 2, "fp32", "diag", 1, 13.5, 26.3),
    ((32, 32, 1), (500, 500, 1), 2, "fp32", "diag", 16, 225.4, 171.0),
]


@pytest.mark.parametrize("box,N,nc,vectors,scene,nrhs,resident,steps", MEASURED)
def test_resident_rhs(driver, box, N, nc, vectors, scene, nrhs, resident, steps):
    """The faster of the two solvers by the number of right-hand sides."""
    pays = run(driver, "pays", *box, *N, nc, int(vectors == "fp64"), int(scene == "mu"), int(scene == "full"), nrhs).strip()
    assert pays == ("1" if resident < steps else "0")


@pytest.mark.parametrize("N,nrhs,narrow,ty_max,reduces,ty,kz,want", [
    ((128, 128, 128), 1, 0, 8, 1, 4, 16, "4 16"),          # as given
    ((203, 180, 151), 1, 0, 8, 1, 1, 1, "1 8"),            # 720 tiles a plane
    ((700, 700, 700), 1, 0, 8, 1, 4, 1, "4 128"),
    ((2, 174763, 1), 1, 1, 8, 0, 4, 1, "4 1"),             # no partial sums: any number of tiles
    ((2, 174763, 1), 1, 1, 8, 1, 4, 1, "8 1"),             # one plane: only rows can grow
    ((2, 174763, 1), 1, 0, 8, 1, 4, 1, "no"),
    ((2, 174763, 1), 1, 0, 4, 1, 4, 16, "no"),
    ((4096, 4096, 1), 1, 0, 8, 1, 4, 1, "no"),
    ((1, 600000, 1), 1, 1, 8, 0, 4, 1, "8 1"),             # rows of tiles beyond a launch's 65,535
    ((1, 1200000, 1), 1, 1, 8, 0, 4, 1, "no"),
    ((16, 16, 200), 5000, 0, 8, 1, 4, 4, "4 16"),          # planes times right-hand sides beyond 65,535
    ((1, 1, 1), 65535, 0, 8, 1, 1, 1, "1 1"),
])
def test_tile_fit(driver, N, nrhs, narrow, ty_max, reduces, ty, kz, want):
    """Tiles of planes too large for the partial sums: the planes were doubled
    without end, to a division by zero."""
    assert run(driver, "fit", *N, nrhs, narrow, ty_max, reduces, ty, kz).strip() == want
