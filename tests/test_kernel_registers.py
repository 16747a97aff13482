"""Registers and scratch memory of the persistent RK5 kernels, from the
metadata of the built library: what decides how many waves a SIMD holds (512
registers a lane) and whether a neuron's arrays live in memory.  The limits are
the ones that the kernels' forms were chosen for (rk5_device.h: kOwn, kCompact,
the register budget)."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "nest-gpu_amd", "libnestgpu_amd.so")
TOOLS = "/opt/rocm/llvm/bin"

# two variables a port / one
TWO = ("AeifCondBeta", "AeifCondAlpha", "AeifPscAlphaMS", "IzhCondBeta")
ONE = "AeifPscExpMS"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """(model, ports, uniform parameters, mode) -> (registers, scratch bytes)"""
    if not os.path.exists(os.path.join(TOOLS, "llvm-objdump")):
        pytest.skip("no ROCm binary tools")
    d = tmp_path_factory.mktemp("code")
    shutil.copy(LIB, d / "lib.so")
    subprocess.run([os.path.join(TOOLS, "llvm-objdump"), "--offloading", "lib.so"], cwd=d, check=True,
                   capture_output=True)
    out = {}
    for f in sorted(os.listdir(d)):
        if not f.endswith("gfx950"):
            continue
        notes = subprocess.run([os.path.join(TOOLS, "llvm-readelf"), "--notes", f], cwd=d, check=True,
                               capture_output=True, text=True).stdout
        for part in notes.split("- .agpr_count:")[1:]:
            m = re.search(r"rk5_persistent_kernelINS_\d+(\w+?)ILi(\d+)EEELb([01])ELi(\d)E", part)
            if not m:
                continue
            regs = int(re.search(r"\.vgpr_count:\s+(\d+)", part).group(1))
            scratch = int(re.search(r"\.private_segment_fixed_size:\s+(\d+)", part).group(1))
            out[(m.group(1), int(m.group(2)), m.group(3) == "1", int(m.group(4)))] = (regs, scratch)
    assert len(out) > 100
    return out


@pytest.mark.parametrize("model", TWO)
def test_two_waves_up_to_eight_ports(kernels, model):
    for (name, ports, uni, mode), (regs, _) in kernels.items():
        if name == model and ports <= 8 and mode == 0 and (name != "IzhCondBeta" or ports != 7):
            assert regs <= 256, (ports, uni, regs)


@pytest.mark.parametrize("model", TWO)
def test_no_arrays_in_scratch(kernels, model):
    # (a few spilled registers are let through)
    for (name, ports, uni, mode), (_, scratch) in kernels.items():
        if name == model and mode == 0 and ports <= 17:
            assert scratch <= 64, (ports, uni, scratch)


def test_one_variable_a_port(kernels):
    for ports in range(1, 17):
        assert kernels[(ONE, ports, False, 0)][0] <= 256, ports


def test_learned_step_sizes_two_waves(kernels):
    for ports in range(1, 6):
        assert kernels[("AeifCondBeta", ports, True, 2)][0] <= 256, ports
