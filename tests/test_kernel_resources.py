"""Registers and scratch memory of the built kernels, from the code object's
own metadata: a kernel that is meant to stay in registers does."""
import glob
import re
import shutil
import subprocess
from pathlib import Path

import pytest

LLVM = Path("/opt/rocm/llvm/bin")
ENGINE = Path(__file__).resolve().parents[1] / "jams_amd" / "lib" / "libjamship.so"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """demangled name -> (VGPRs, spilled VGPRs, scratch bytes per lane)"""
    if not (LLVM / "llvm-objdump").exists() or not shutil.which("c++filt") or not ENGINE.exists():
        pytest.skip("needs the LLVM tools and the built engine")
    so = tmp_path_factory.mktemp("code") / ENGINE.name
    shutil.copy(ENGINE, so)
    subprocess.run([LLVM / "llvm-objdump", "--offloading", so], check=True, capture_output=True,
                   cwd=so.parent)
    out = {}
    for code in glob.glob(str(so) + "*gfx950*"):
        notes = subprocess.run([LLVM / "llvm-readelf", "--notes", code], check=True,
                               capture_output=True, text=True).stdout.split(".agpr_count:")[1:]
        names = [re.search(r"\.name:\s+(\S+)", p).group(1) for p in notes]
        plain = subprocess.run(["c++filt"], input="\n".join(names), check=True,
                               capture_output=True, text=True).stdout.splitlines()
        for name, p in zip(plain, notes):
            out[name] = tuple(int(re.search(rf"\.{k}:\s+(\d+)", p).group(1)) for k in
                              ("vgpr_count", "vgpr_spill_count", "private_segment_fixed_size"))
    assert len(out) > 100
    return out


@pytest.mark.parametrize("pattern", [
    # <precision, diagonal, phase, general local terms, cells per lane, one class>:
    # the predictors with the general terms keep five waves and spill
    r"k_heun_ln<\d, \w+, 0, false, ", r"k_heun_ln<\d, \w+, 1, ",
    r"k_heun<", r"k_heun_many<", r"k_rk4<", r"k_dip_(x_fused|zy_fwd|zy_inv)<"])
def test_no_spills(kernels, pattern):
    found = {n: k for n, k in kernels.items() if re.search(pattern, n)}
    assert found
    assert not {n: k for n, k in found.items() if k[1] or k[2]}


def test_persistent_step_copies_no_parameters(kernels):
    """its parameters are about 400 bytes; spilled scalars take less than 100"""
    found = {n: k for n, k in kernels.items() if "k_heun_step<" in n}
    assert found and all(k[1] == 0 for k in found.values())
    assert not {n: k for n, k in found.items() if k[2] > 100}


@pytest.mark.parametrize("pattern,most", [
    # <FP64, rows of full tensors by pattern, no general terms, ...>: six waves
    (r"k_rk4<0, 6, false, ", 80),
    # <FP32 field, pair programs with DMI, phase, no general terms, one class>:
    # seven and five waves
    (r"k_heun<1, 12, 0, false, 2>", 72), (r"k_heun<1, 12, 1, false, 2>", 96)])
def test_full_tensors_leave_room_for_other_waves(kernels, pattern, most):
    found = {n: k for n, k in kernels.items() if re.search(pattern, n)}
    assert found and all(k[0] <= most for k in found.values())
