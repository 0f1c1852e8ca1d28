"""The three-operation quotient of the nonlinear momentum kernels
(gpu-comcot_amd/csrc/fastdiv.h), on the host: for every divisor, every
numerator whose quotient lies close enough to a rounding midpoint to be
rounded wrongly gives the IEEE quotient.  The device's refined reciprocal,
which the proof takes as 1/b rounded to nearest, and random pairs are
checked on the GPU in tests/test_gpu_fastdiv.py."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_quotients_near_midpoints(tmp_path):
    exe = tmp_path / "quotient_check"
    flags = ["-O2", "-ffp-contract=off", "-fopenmp"]
    if "fma" in open("/proc/cpuinfo").read().split():
        flags.append("-mfma")
    subprocess.run(["g++", *flags, os.path.join(HERE, "quotient_check.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True,
                         env=dict(os.environ, OMP_NUM_THREADS=str(min(8, os.cpu_count() or 1))))
    tried, bad = (int(v) for v in out.stdout.split())
    assert bad == 0
    assert tried > 2.5e8  # 24 numerators a divisor, and some 90 M near midpoints
