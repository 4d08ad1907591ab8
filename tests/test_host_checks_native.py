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
    pays = run(driver, "pays", *box, *N, nc, int(vectors == "fp64"), int(scene == "mu"), int(scene == "full"), nrhs, 512 if nrhs == 1 else 32).strip()
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


@pytest.mark.parametrize("box,N,nrhs,steps,resident", [
    ((8, 8, 4), (40, 40, 40), 2, 1, 0),     # 104 against 62 µs a step (step by step), the start of each launch
    ((8, 4, 4), (20, 20, 20), 2, 1, 0),     # 52 against 47
    ((8, 4, 4), (20, 20, 20), 2, 8, 1),
    ((8, 4, 4), (20, 20, 20), 1, 512, 1),   # one right-hand side: up to 512 steps a launch whatever the chunk
])
def test_resident_short_launches(driver, box, N, nrhs, steps, resident):
    assert int(run(driver, "pays", *box, *N, 3, 1, 0, 0, nrhs, steps)) == resident


# A on one right-hand side (three: last column): µs per apply by (rows, planes) of a tile, measured; the
# three fastest and 4 × 16
APPLIES = [
    ((64, 64, 64), "mu", "fp32", 1, {(8, 2): 25.4, (4, 2): 26.2, (8, 3): 27.3, (4, 16): 57.0}),
    ((70, 66, 72), "mu", "fp32", 1, {(4, 5): 34.6, (8, 6): 35.0, (4, 6): 36.7, (4, 16): 58.5}),
    ((56, 100, 41), "mu", "fp32", 3, {(8, 7): 38.2, (4, 7): 38.7, (8, 8): 41.0, (4, 16): 57.4}),
    ((96, 90, 100), "mu", "fp32", 1, {(8, 10): 47.0, (4, 10): 49.1, (8, 11): 49.7, (4, 16): 66.6}),
    ((128, 128, 128), "diag", "fp64", 1, {(4, 16): 78.3, (4, 17): 81.5, (8, 16): 82.5}),
    ((128, 128, 128), "diag", "fp32", 1, {(4, 11): 56.6, (4, 12): 58.3, (4, 13): 59.9, (4, 16): 61.0}),
    ((110, 112, 90), "full", "fp64", 1, {(4, 10): 72.1, (8, 10): 74.5, (4, 11): 77.1, (4, 16): 92.7}),
    ((150, 60, 170), "mu", "fp64", 1, {(4, 16): 90.8, (4, 8): 92.7, (4, 5): 93.7}),
    ((150, 60, 170), "hee", "fp32", 1, {(4, 10): 52.8, (4, 11): 55.2, (4, 12): 57.7, (4, 16): 61.9}),
    ((190, 33, 120), "mu", "fp64", 1, {(4, 7): 44.7, (4, 8): 46.3, (8, 8): 47.2, (4, 16): 60.3}),
    ((181, 62, 89), "mu", "fp32", 1, {(8, 9): 46.3, (4, 9): 47.6, (8, 10): 48.4, (4, 16): 66.7}),
    ((27, 172, 92), "hee", "fp64", 1, {(8, 9): 39.5, (4, 9): 40.8, (8, 10): 41.6, (4, 16): 56.9}),
]


@pytest.mark.parametrize("N,scene,vectors,nrhs,us", APPLIES)
def test_apply_tiles(driver, N, scene, vectors, nrhs, us):
    """The rule's tile is one of the fastest three, within 4 % of the fastest."""
    narrow = scene == "diag" and 64 * -(-N[0] // 64) > 32 * -(-N[0] // 32)
    pick = run(driver, "tile", *N, nrhs, int(vectors == "fp64"), 1, int(scene == "mu"), int(scene == "full"), 0,
               int(scene == "hee"), 0, int(narrow), 0)
    pick = tuple(map(int, pick.split()))
    assert pick in us and us[pick] <= 1.04 * min(us.values())


def test_scal_store(driver):
    """The lead block of a resident launch stores the scalars without the mark that
    a block which gave up waiting may set meanwhile."""
    assert "scal ok" in run(driver, "scal")


# COCG's fused step: µs by (rows, planes), measured; the three fastest and 4 × 16
COCG = [
    ((64, 64, 64), "fp64", 1, {(4, 4): 54.1, (4, 3): 54.7, (8, 3): 56.2, (4, 16): 97.1}),
    ((70, 66, 72), "fp64", 3, {(4, 15): 139.9, (4, 16): 146.5, (4, 8): 146.8, (4, 9): 151.1}),
    ((70, 66, 72), "fp32", 1, {(4, 5): 57.0, (4, 6): 61.2, (8, 6): 64.1, (4, 16): 96.5}),
    ((100, 90, 96), "fp32", 1, {(4, 9): 82.8, (4, 10): 86.2, (8, 10): 89.7, (4, 16): 113.6}),
    ((150, 60, 170), "fp64", 1, {(4, 16): 228.7, (8, 18): 231.2, (4, 18): 239.8}),
    ((150, 60, 170), "fp32", 1, {(4, 16): 146.2, (4, 18): 155.6, (4, 8): 156.2}),
    ((30, 170, 60), "fp64", 1, {(4, 6): 60.8, (8, 6): 63.9, (4, 7): 64.4, (4, 16): 91.6}),
]


@pytest.mark.parametrize("N,vectors,nrhs,us", COCG)
def test_cocg_tiles(driver, N, vectors, nrhs, us):
    pick = run(driver, "tile", *N, nrhs, int(vectors == "fp64"), 0, 0, 0, 0, 0, 0, 0, 1)
    pick = tuple(map(int, pick.split()))
    assert pick in us and us[pick] <= 1.07 * min(us.values())
