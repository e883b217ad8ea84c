"""The detector's transforms keep everything in registers and LDS: no kernel of
theirs has private memory (a choice between two complex values once put the
FP64 forward rows' elements there).  Reads the metadata of the object that the
build left; CPU only.
"""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
OBJ = os.path.join(ROOT, "bimsim-cuda_amd", "_build", "detector.o")
LLVM = "/opt/rocm/llvm/bin"


@pytest.mark.skipif(not os.path.exists(OBJ) or not shutil.which("objcopy") or
                    not os.path.exists(os.path.join(LLVM, "llvm-readelf")),
                    reason="needs a build and the LLVM tools")
def test_detector_kernels_have_no_private_memory(tmp_path):
    bundle, co = str(tmp_path / "fatbin"), str(tmp_path / "code.o")
    subprocess.run(["objcopy", "-O", "binary", "--only-section=.hip_fatbin", OBJ, bundle], check=True)
    subprocess.run([os.path.join(LLVM, "clang-offload-bundler"), "--unbundle", "--type=o",
                    "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--input={bundle}",
                    f"--output={co}"], check=True)
    notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", co], check=True,
                           capture_output=True, text=True).stdout
    names = re.findall(r"^\s+\.name:\s+(_Z\S+)$", notes, re.M)
    sizes = [int(v) for v in re.findall(r"\.private_segment_fixed_size:\s+(\d+)", notes)]
    assert len(names) == len(sizes) > 100
    bands = [(n, s) for n, s in zip(names, sizes) if re.search(r"(rows_fwd|cols_band|rows_inv)", n)]
    assert len(bands) > 80
    assert [n for n, s in bands if s] == []
