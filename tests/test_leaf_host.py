"""The four-wide walk's node and leaf records against the forms they stand
for, compiled on the host with g++ (no GPU)."""

import ctypes as C
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def leafcheck(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    out = tmp_path_factory.mktemp("leaf") / "leafcheck.so"
    subprocess.run(["g++", "-O2", "-shared", "-fPIC", "-std=c++17", "-pthread", f"-I{ROOT / 'pyradiance_amd/csrc'}",
                    str(ROOT / "tests/native/leaf_check.cpp"), str(ROOT / "pyradiance_amd/csrc/rg_bvh.cpp"),
                    "-o", str(out)], check=True)
    L = C.CDLL(str(out))
    L.check_quantized.argtypes = [C.c_int, C.c_uint, C.c_int, C.c_double]
    L.check_leaf.argtypes = [C.c_int, C.c_int, C.c_uint, C.c_int, C.c_int, C.POINTER(C.c_long)]
    L.check_leaf.restype = C.c_long
    L.check_walk_boxes.argtypes = [C.c_int, C.c_int, C.c_uint, C.c_double, C.c_double, C.c_int]
    L.check_walk_boxes.restype = C.c_long
    L.check_walk_nan.argtypes = [C.c_int, C.c_uint]
    L.check_order.argtypes = [C.c_int, C.c_int, C.c_uint, C.c_int, C.POINTER(C.c_long)]
    return L


@pytest.mark.parametrize("n,nused,far", [(1, 2, 1.0), (40000, 2, 10.0), (40000, 3, 1e3), (40000, 4, 10.0), (40000, 4, 1e5)])
def test_rounded_boxes_hold_the_boxes_they_stand_for(leafcheck, n, nused, far):
    assert leafcheck.check_quantized(n, 5, nused, far) == 0


@pytest.mark.parametrize("nv,degenerate", [(3, 0), (4, 0), (3, 1), (4, 1), (4, 2), (5, 0)])
def test_leaf_records_hit_what_the_primitive_tables_hit(leafcheck, nv, degenerate):
    hits = C.c_long()
    assert leafcheck.check_leaf(2000, 500, 17, nv, degenerate, C.byref(hits)) == 0
    assert hits.value > 100000


@pytest.mark.parametrize("n,grid", [(2, 0), (3, 0), (5, 1), (300, 0), (300, 1), (5000, 0)])
def test_ties_are_ordered_as_a_walk_of_the_unrounded_boxes(leafcheck, n, grid):
    pairs = C.c_long()
    assert leafcheck.check_order(n, 200 if n > 100 else 200000, 23, grid, C.byref(pairs)) == 0
    assert pairs.value > 0


@pytest.mark.parametrize("ext", [0.05, 6.0, 2000.0])
@pytest.mark.parametrize("far,flat", [(0.0, 0), (0.0, 1), (8.0, 0), (8.0, 1)])
def test_walk_enters_the_boxes_its_ray_meets(leafcheck, ext, far, flat):
    """In FP32 (u = 2^-24) a plane's distance is off by at most u (4 |plane| +
    4 |origin| + |plane - origin| + 3 node side + |plane - origin|) measured
    along its axis: u (12 ext / 2 + 6 (far + 1/2) ext) = 3.4e-6 ext at far = 8,
    inside the 4e-6 ext + 1e-5 that boxes are widened by."""
    assert leafcheck.check_walk_boxes(2000, 200, 31, ext, far, flat) == 0


def test_walk_enters_nothing_for_rays_that_are_not_numbers(leafcheck):
    assert leafcheck.check_walk_nan(20000, 37) == 0
