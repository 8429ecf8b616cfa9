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
