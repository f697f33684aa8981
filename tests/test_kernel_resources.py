"""What the compiler made of the kernels, read from the metadata of the library that was built from them."""
import glob
import os
import re
import shutil
import subprocess

import pytest

LLVM = "/opt/rocm/llvm/bin"
LIBRARY = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nnfusion_amd", "lib", "libnnf_hip_kernels.so")


# The row-streaming kernels keep their activations in registers from the first weight to the last: one that spills them takes twice its
# time (RMSNorm at K = 8192, where the sums of squares had been moved behind the last block of activations: 9 rows x 4096 26 us, 13 without).
def test_row_streaming_kernels_use_no_private_memory(tmp_path):
    if not os.path.exists(os.path.join(LLVM, "llvm-objdump")) or not os.path.exists(LIBRARY):
        pytest.skip("needs the built library and the ROCm LLVM tools")
    lib = shutil.copy(LIBRARY, tmp_path / "lib.so")
    subprocess.run([os.path.join(LLVM, "llvm-objdump"), "--offloading", str(lib)], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    seen, spilled = 0, []
    for code_object in glob.glob(str(tmp_path / "lib.so.*gfx950*")):
        notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", code_object], check=True, capture_output=True, text=True).stdout
        for name, private in re.findall(r"\.name:\s+(_Z\S+)\n\s+\.private_segment_fixed_size:\s+(\d+)", notes):
            if "mrows" in name or "gemv_rows" in name:
                seen += 1
                if int(private):
                    spilled.append((name, int(private)))
    assert seen > 100
    assert not spilled
