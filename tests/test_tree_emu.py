"""CPU: a single layer tree (tree.hip) against the runtime emulator of
tests/batch_emu, compiled with g++ (AddressSanitizer and UBSan on): which forms
its launches take, the device memory that its layers report, and that every
sub-step of a nest finds its boundary fluxes made."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
EMU = os.path.join(HERE, "batch_emu")
CSRC = os.path.join(os.path.dirname(HERE), "gpu-comcot_amd", "csrc")


@pytest.fixture(scope="module")
def emu_tree(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path_factory.mktemp("tree_emu") / "emu_tree")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined",
                    "-fno-omit-frame-pointer", "-I", EMU, "-I", CSRC, "-x", "c++",
                    os.path.join(CSRC, "tree.hip"), os.path.join(CSRC, "batch.hip"), "-x", "none", os.path.join(EMU, "emu_runtime.cpp"),
                    os.path.join(EMU, "emu_kernels.cpp"), os.path.join(EMU, "emu_tree.cpp"), "-o", exe],
                   check=True, capture_output=True, text=True)
    return exe


@pytest.mark.parametrize("check", ["tuned-fallback", "footprint", "substeps"])
def test_tree(emu_tree, check):
    r = subprocess.run([emu_tree, check], capture_output=True, text=True, timeout=120,
                       env=dict(os.environ, ASAN_OPTIONS="detect_leaks=1"))
    assert r.returncode == 0, r.stderr[-2000:]
