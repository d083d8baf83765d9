"""Registers of the GEMM kernels that count, read from the built library: a consumer's wavefront (64 registers) has to fit
on the SIMD beside theirs, or a consumer that polls on every CU keeps the GEMM it waits for from starting."""
import os
import re
import shutil
import subprocess

import pytest

from flashoverlap_amd import _capi, build

LLVM = os.path.join(os.path.dirname(os.path.dirname(build.HIPCC)), "llvm", "bin")
SIMD, CONSUMER = 512, 64


def test_a_consumer_fits_beside_the_kernels_that_count(tmp_path):
    if not os.path.exists(os.path.join(LLVM, "llvm-readelf")):
        pytest.skip("no llvm-readelf beside hipcc")
    shutil.copy2(_capi.KERNEL_LIB, tmp_path / "lib.so")
    subprocess.run([os.path.join(LLVM, "llvm-objdump"), "--offloading", "lib.so"], cwd=tmp_path, check=True,
                   stdout=subprocess.DEVNULL)
    seen = 0
    for part in sorted(p for p in os.listdir(tmp_path) if p.endswith(build.ARCH)):
        notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", part], cwd=tmp_path, check=True,
                               capture_output=True, text=True).stdout
        # one kernel's entries stand in alphabetical order, .name in front of .vgpr_count
        for name, rest in re.findall(r"\.name: +(\S+)\n(.*?\.vgpr_spill_count: +\d+)", notes, re.S):
            tile = re.search(r"fo_gemm_tile_kernelI\w+_tag(?:Li\d+E){4}Li(\d)E", name)
            large = re.search(r"fo_gemm256_kernelI\w+_tagLi(\d)E", name)
            mode = tile or large
            if not mode or int(mode.group(1)) not in (1, 2):  # the signal and scatter epilogues
                continue
            registers = int(re.search(r"\.vgpr_count: +(\d+)", rest).group(1))
            waves = 2 if tile else 1
            assert waves * -(-registers // 8) * 8 + CONSUMER <= SIMD, (name, registers)
            assert int(re.search(r"\.vgpr_spill_count: +(\d+)", rest).group(1)) == 0, name
            seen += 1
    assert seen == 2 * 2 * (11 + 8 + 1)  # types, epilogues; tiles, their shifted forms, the 256x256 kernel


def test_the_kernel_that_consumes_and_normalises_fits_beside_the_signalling_gemm(tmp_path):
    if not os.path.exists(os.path.join(LLVM, "llvm-readelf")):
        pytest.skip("no llvm-readelf beside hipcc")
    shutil.copy2(_capi.KERNEL_LIB, tmp_path / "lib.so")
    subprocess.run([os.path.join(LLVM, "llvm-objdump"), "--offloading", "lib.so"], cwd=tmp_path, check=True,
                   stdout=subprocess.DEVNULL)
    gemm, rows = [], []
    for part in sorted(p for p in os.listdir(tmp_path) if p.endswith(build.ARCH)):
        notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", part], cwd=tmp_path, check=True,
                               capture_output=True, text=True).stdout
        for name, rest in re.findall(r"\.name: +(\S+)\n(.*?\.vgpr_spill_count: +\d+)", notes, re.S):
            registers = -(-int(re.search(r"\.vgpr_count: +(\d+)", rest).group(1)) // 8) * 8
            if re.search(r"fo_gemm256_kernelI\w+_tagLi1E", name):
                gemm.append(registers)
            if re.search(r"fo_norm_rows_kernelI\w+_tagLi\dELb\dELi\dELb1E", name):
                rows.append(registers)
                assert int(re.search(r"\.vgpr_spill_count: +(\d+)", rest).group(1)) == 0, name
    assert len(gemm) == 2 and len(rows) == 2 * 2 * 4  # types, cache policies, chunks a lane
    assert max(gemm) + max(rows) <= SIMD


def test_what_runs_beside_the_earlier_waves_fits_beside_the_kernels_that_sum_the_last(tmp_path):
    """The signal and scatter epilogues with the last wave's sums: a consumer's wavefront beside both, and beside the first the
    kernel that consumes and normalises (128 registers)."""
    if not os.path.exists(os.path.join(LLVM, "llvm-readelf")):
        pytest.skip("no llvm-readelf beside hipcc")
    shutil.copy2(_capi.KERNEL_LIB, tmp_path / "lib.so")
    subprocess.run([os.path.join(LLVM, "llvm-objdump"), "--offloading", "lib.so"], cwd=tmp_path, check=True,
                   stdout=subprocess.DEVNULL)
    seen = 0
    for part in sorted(p for p in os.listdir(tmp_path) if p.endswith(build.ARCH)):
        notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", part], cwd=tmp_path, check=True,
                               capture_output=True, text=True).stdout
        for name, rest in re.findall(r"\.name: +(\S+)\n(.*?\.vgpr_spill_count: +\d+)", notes, re.S):
            mode = re.search(r"fo_gemm256_kernelI\w+_tagLi([56])E", name)
            if not mode:
                continue
            registers = -(-int(re.search(r"\.vgpr_count: +(\d+)", rest).group(1)) // 8) * 8
            assert registers + (128 if mode.group(1) == "5" else CONSUMER) <= SIMD, (name, registers)
            assert int(re.search(r"\.vgpr_spill_count: +(\d+)", rest).group(1)) == 0, name
            seen += 1
    assert seen == 4
