"""The bound below which Manning friction leaves a flux as it is (drag_vanishes,
gpu-comcot_amd/csrc/fastdiv.h), on the host: where it holds, both friction
terms return the flux bit for bit."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_skipped_friction_would_not_move_the_flux(tmp_path):
    exe = tmp_path / "friction_check"
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", os.path.join(HERE, "friction_check.cpp"),
                    "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
    held, moved = (int(v) for v in out.split())
    assert moved == 0
    assert held > 1000000


def test_skipped_friction_would_not_move_the_flux_out_of_range(tmp_path):
    exe = tmp_path / "friction_overflow_check"
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off",
                    os.path.join(HERE, "friction_overflow_check.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
    held, moved = (int(v) for v in out.split())
    assert moved == 0
    assert held > 1000
