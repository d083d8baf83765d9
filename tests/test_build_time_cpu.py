"""The K step of the 256x256 GEMM kernel is laid out before the optimiser starts: as loops for it to unroll, the library's
ten instantiations cost half an hour of CPU time."""
import os
import resource
import shutil
import subprocess

import pytest

from flashoverlap_amd import build


def test_an_instantiation_compiles_quickly(tmp_path):
    """3 s of CPU time; laid out by the optimiser 165."""
    if not shutil.which(build.HIPCC):
        pytest.skip("no hipcc")
    before = resource.getrusage(resource.RUSAGE_CHILDREN).ru_utime
    subprocess.run([build.HIPCC] + build.HIP_FLAGS + ["--cuda-device-only", "-w", "-DFO_INST_DTYPE=0", "-DFO_INST_MODE=1", "-c",
                    os.path.join(build.CSRC, "fo_gemm256_inst.hip"), "-o", str(tmp_path / "x.o")], check=True,
                   stderr=subprocess.DEVNULL)
    assert resource.getrusage(resource.RUSAGE_CHILDREN).ru_utime - before < 30
