"""Host decisions of the launches (CPU only, no kernel runs)."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
STATIC_SCRATCH = 64 << 20


@pytest.fixture(scope="module")
def shapes(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ is not available")
    exe = str(tmp_path_factory.mktemp("shapes") / "launch_shapes")
    pkg = os.path.join(ROOT, "ctsim_amd")
    r = subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{ROOT}/include", f"-I{pkg}/csrc",
                        f"-I{ROCM}/include", os.path.join(ROOT, "tests", "cxx", "launch_shapes.cpp"), "-o", exe,
                        f"-L{pkg}", "-lctsim_amd", f"-Wl,-rpath,{pkg}", f"-L{ROCM}/lib", "-lamdhip64",
                        f"-Wl,-rpath,{ROCM}/lib"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr

    def run(*args):
        out = subprocess.run([exe, *map(str, args)], capture_output=True, text=True, timeout=60)
        assert out.returncode == 0, out.stderr
        return out.stdout.split()
    return run


@pytest.mark.parametrize("method", ["fft", "convolution"])
@pytest.mark.parametrize("geom", [0, 1, 2])
@pytest.mark.parametrize("nx,nView", [(900, 901), (960, 961), (1000, 1001), (1100, 1101), (1200, 1201), (1300, 1301),
                                      (1300, 1138), (1500, 255), (1700, 130), (1024, 1024), (2048, 250)])
def test_whole_slices_keep_the_rules_kernel(shapes, geom, nx, nView, method):
    """A slice that only its view groups' partial images keep from fitting the
    static scratch runs with fewer groups, not with another kernel."""
    w = shapes("slice", geom, min(2048, nx + nx // 10), nView, nx, nx, method, "linear")
    rule, used = list(map(int, w[1:5])), list(map(int, w[6:10]))
    scratch, default = int(w[11]), int(w[13])
    assert used[:3] == rule[:3]
    assert used[3] == rule[3] or (used[3] < rule[3] and scratch <= STATIC_SCRATCH)
    if default <= STATIC_SCRATCH:
        assert scratch <= STATIC_SCRATCH


@pytest.mark.parametrize("interp", ["linear", "cubic"])
@pytest.mark.parametrize("geom", [0, 1, 2])
@pytest.mark.parametrize("nx,ny,nDet,nView", [(103, 1980, 1790, 2655), (111, 805, 1141, 943), (158, 611, 1170, 1025),
                                              (217, 1396, 1944, 2624), (96, 536, 499, 1042), (142, 714, 1150, 1182)])
def test_tall_images_take_narrow_tiles(shapes, geom, interp, nx, ny, nDet, nView):
    """Columns much wider than rows are high: tiles of 16 columns, whose
    windows are the shorter ones."""
    w = shapes("slice", geom, nDet, nView, nx, ny, "fft", interp)
    lanes, windows = int(w[3]), list(map(int, w[15:18]))
    full = nDet + 4
    rule, eight, sixteen = (x if x > 0 else full for x in windows)
    assert 1.2 * sixteen < eight
    assert lanes == 16
    assert rule <= sixteen


@pytest.mark.parametrize("geom", [0, 2])
@pytest.mark.parametrize("nx,ny,nDet,nView", [(138, 407, 567, 462), (148, 148, 316, 269), (149, 149, 319, 334),
                                              (171, 171, 235, 442), (301, 301, 622, 730), (432, 432, 791, 515)])
def test_small_linear_slices_take_the_plain_kernel(shapes, geom, nx, ny, nDet, nView):
    """A parallel or equilinear linear update costs less than the mirror
    kernel's staging on images this small."""
    w = shapes("slice", geom, nDet, nView, nx, ny, "fft", "linear")
    assert int(w[1]) == 0


@pytest.mark.parametrize("nx,nView,method", [(423, 1516, "convolution")])
def test_fewer_groups_leave_enough_workgroups(shapes, nx, nView, method):
    """Where the static scratch leaves the mirror kernel too few workgroups,
    the plain kernel's smaller share of the views fills the chip."""
    w = shapes("slice", 0, 1606, nView, nx, 932, method, "linear")
    assert int(w[1]) == 3 and int(w[6]) == 0
    assert int(w[11]) <= STATIC_SCRATCH


@pytest.mark.parametrize("angles,largest,covered", [("0 1 -27.9 3", "27.9", 1), ("0 28", "28", 0), ("-1000 1", "1000", 0),
                                                    ("1000 nan 1", "nan", 0), ("nan", "nan", 0), ("1 nan", "nan", 0),
                                                    ("inf nan 2", "nan", 0), ("1 -inf", "inf", 0)])
def test_fan_bounds_see_every_angle(shapes, angles, largest, covered):
    """An angle that is no number hides no larger one from the FP64 fan-beam
    kernel's condition."""
    got = shapes("fan64", *angles.split())
    assert got[0].lstrip("-") == largest and int(got[1]) == covered


@pytest.mark.parametrize("args,short", [
    ("equiangular 1024 1440 2 2 64 4 0 0", 1), ("parallel 367 320 2 2 8 2 0 0", 1), ("equiangular 33 10 2 2 8 2 0 0", 1),
    # few parallel rays, some of them along a rectangle's side
    ("parallel 33 10 2 2 1 2 0 0", 0), ("parallel 64 64 2 2 1 2 0 0", 0), ("parallel 33 40 2 2 64 2 0 0", 1),
    # other types: in few of many items, in most items, in a scan that the chip holds at once
    ("equilinear 1024 1440 2 2 64 2 1 0.1", 1), ("equilinear 1024 1440 2 2 64 2 10 0.2", 0),
    ("equilinear 367 320 2 2 64 2 1 0.03", 0), ("equiangular 1024 1440 2 2 herman", 0),
    ("equiangular 1024 1440 2 2 shepp-logan", 1),
    # ends of rays in the elements' disc
    ("equiangular 1024 720 2 1 8 2 0 0", 0), ("equilinear 1024 720 2 1 8 2 0 0", 1),
    ("equilinear 1024 720 2 0.9 8 2 0 0", 0), ("parallel 1024 720 0.9 2 8 2 0 0", 0), ("parallel 1024 720 1 1 8 2 0 0", 1)])
def test_short_ray_sums_where_they_pay(shapes, args, short):
    assert shapes("scan", *args.split()) == [str(short)]
