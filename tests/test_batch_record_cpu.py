"""The records from which a batch chooses its kernels (chroma_amd/csrc/batch.cpp), on the CPU: launches that need
different kernels must differ in their keys, or one problem's kernel would run on the records of another."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CLANG = "/opt/rocm/llvm/bin/clang++"


@pytest.fixture(scope="module")
def lines(tmp_path_factory):
    if not os.path.exists(CLANG):
        pytest.skip("ROCm clang is not installed")
    lib = os.path.join(ROOT, "chroma_amd")
    exe = str(tmp_path_factory.mktemp("record") / "record_check")
    subprocess.run([CLANG, "-std=c++17", "-x", "hip", "--cuda-host-only", "-nogpulib", "--offload-arch=gfx950",
                    "-I/opt/rocm/include", "-I", os.path.join(ROOT, "include"), "-I", os.path.join(lib, "csrc"),
                    os.path.join(HERE, "record_check.cpp"), "-L", lib, "-lchroma_mi355x",
                    "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath," + lib, "-Wl,-rpath,/opt/rocm/lib", "-o", exe],
                   check=True, timeout=300)
    out = subprocess.run([exe], capture_output=True, text=True, check=True, timeout=60).stdout
    return [ln.split() for ln in out.splitlines()]


def test_tails_have_their_own_keys(lines):
    keys = [tuple(ln[2:]) for ln in lines if ln[0] == "key"]
    assert len(keys) == 5 and len(set(keys)) == 5, keys


def test_default_shapes_by_size(lines):
    """Untuned launch shapes (block, tiled, kernel) on both sides of the sizes where the rules change."""
    got = {tuple(int(v) for v in ln[1:5]): tuple(int(v) for v in ln[5:]) for ln in lines if ln[0] == "shape"}
    D, S, H = 0, 1, 2
    for prec in (D, S):
        assert got[16, 32, prec, 0] == (64, 0, 5)  # direction-split
    assert got[16, 32, H, 0] == (64, 1, 1)
    for prec in (D, S, H):
        assert got[32, 64, prec, 0] == (64, 1, 3)  # slabs
        for lat in ((48, 96), (64, 48)):  # round-robin, a ninth of the lanes idle on 48 x 48 planes
            assert got[lat + (prec, 0)] == got[lat + (prec, 1)] == (256, 0, 3)
    # time slices of 23328 and 32000 sites: round-robin for the FP64 operator alone
    assert got[36, 60, D, 0] == (256, 0, 3) and got[40, 60, D, 0] == (128, 0, 3)
    for prec, which in ((D, 1), (S, 0), (H, 0), (H, 1)):
        assert got[40, 60, prec, which] == (64, 0, 3)
