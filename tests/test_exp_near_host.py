"""The clampless exponential of the reciprocal right-hand sides
(stepfactor.h exp_fma_near) gives exp_fma's bits over the range it is used on."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_exp_near_is_exp(tmp_path):
    exe = tmp_path / "exp_near_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-mfma", "-ffp-contract=off",
                    os.path.join(ROOT, "tests", "host", "exp_near_check.cpp"), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "0", r.stdout
