"""Registers of kernels whose workgroups have to fit beside each other, as the compiler left them in the built library."""

from __future__ import annotations

import re
import shutil
import subprocess
from pathlib import Path

import pytest

TOOLS = Path("/opt/rocm/llvm/bin")


@pytest.fixture(scope="module")
def registers(tmp_path_factory):
    """{kernel's mangled name: (registers a lane, of them spilled)}"""
    from paged_llm_rs_amd import build, kernels

    if not all((TOOLS / tool).exists() for tool in ("llvm-objdump", "llvm-readelf")):
        pytest.skip("no LLVM tools to read the library's notes with")
    kernels.library()
    folder = tmp_path_factory.mktemp("objects")
    shutil.copy(build.library_path("hip"), folder / "lib.so")
    subprocess.run([str(TOOLS / "llvm-objdump"), "--offloading", "lib.so"], cwd=folder, check=True, capture_output=True)
    found = {}
    for part in folder.glob("lib.so.*gfx950*"):
        notes = subprocess.run([str(TOOLS / "llvm-readelf"), "--notes", str(part)], check=True, capture_output=True, text=True).stdout
        for kernel in notes.split("- .agpr_count:")[1:]:
            name = re.search(r"^ +\.symbol: +(\S+)\.kd", kernel, re.M).group(1)
            found[name] = tuple(int(re.search(rf"^ +\.{which}: +(\d+)", kernel, re.M).group(1)) for which in ("vgpr_count", "vgpr_spill_count"))
    return found


def _of(registers, pattern):
    some = {name: counts for name, counts in registers.items() if re.search(pattern, name)}
    assert some, f"no kernel {pattern}"
    return some


def test_two_workgroups_of_single_tokens_attention_fit_a_compute_unit(registers):
    """Four waves a workgroup and 512 registers a lane of a unit of execution: 256 for each, without sinks, slopes and further extras (the last of the
    template's arguments) and with the first two of them.  With 257 a second engine's launches wait for the first's."""
    for name, (used, spilled) in _of(registers, r"paged_attention_decode_kernelI(Li\d+E){4}Li[01]E").items():
        assert used <= 256 and spilled == 0, (name, used, spilled)


def test_two_workgroups_of_a_chain_fit_a_compute_unit_without_spills(registers):
    """And of the 32-bit one, of eight waves, whose bound of 128 two or three values do not fit."""
    for name, (used, spilled) in _of(registers, r"gemm_chain_kernel").items():
        assert used <= 256 and spilled == 0, (name, used, spilled)
    for name, (used, spilled) in _of(registers, r"gemm_chain_f32_kernel").items():
        assert used <= 128 and spilled <= 3, (name, used, spilled)
