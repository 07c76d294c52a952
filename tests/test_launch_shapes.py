"""Host decisions of the backprojection launches (CPU only, no kernel runs)."""
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
