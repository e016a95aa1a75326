"""Registers and LDS of kernels whose time they decide, as the compiler
reports them with the library's own flags."""
import os
import re
import shutil
import subprocess

import pytest

from libclsph_amd import build

pytestmark = pytest.mark.skipif(not shutil.which(build.HIPCC), reason="needs hipcc")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """The report of each kernel of sph.hip, by its mangled name."""
    flags = [f for f in build.FLAGS if f != "-shared"]
    r = subprocess.run([build.HIPCC] + flags +
                       ["--cuda-device-only", "-c", os.path.join(build.CSRC, "sph.hip"), "-o",
                        str(tmp_path_factory.mktemp("res") / "sph.o"),
                        "-Rpass-analysis=kernel-resource-usage"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return dict(re.findall(r"Function Name: (\S+)(.*?)(?=Function Name|\Z)", r.stderr, re.S))


def test_overflow_forces_leave_most_waves_in_flight(kernels):
    """Nearly every wave of the overflow kernel reads its counts and leaves:
    at least seven of them per SIMD (72 of its 512 registers), none spilled.
    At three, a macro step of 1,048,576 particles waited 7.1 us for it instead
    of 4.5."""
    found = [k for k in kernels if "k_forces_overflow" in k or "k_forcesILb1E" in k]
    assert len(found) == 1
    report = kernels[found[0]]
    assert int(re.search(r" VGPRs: (\d+)", report).group(1)) <= 72
    assert int(re.search(r"ScratchSize \[bytes/lane\]: (\d+)", report).group(1)) == 0


def test_density_staging_fills_half_a_compute_unit(kernels):
    """Two 512-thread density work-groups share a compute unit's 160 KB of
    LDS, and stage as many candidates (16 bytes) as their halves hold."""
    (name,) = [k for k in kernels if "k_densityILi8E" in k]
    lds = int(re.search(r"LDS Size \[bytes/block\]: (\d+)", kernels[name]).group(1))
    assert 81920 - 128 < lds <= 81920


@pytest.mark.parametrize("waves", [2, 4])
def test_smaller_work_groups_stage_two_cells_per_wave(kernels, waves):
    """768 candidates per wave (16 bytes) and the offsets of the 64 half-cells
    around each of two cells per wave."""
    (name,) = [k for k in kernels if f"k_densityILi{waves}E" in k]
    lds = int(re.search(r"LDS Size \[bytes/block\]: (\d+)", kernels[name]).group(1))
    assert lds >= 16 * 768 * waves + 4 * (64 * 2 * waves + 1)
