"""The general kernel's step loop keeps its values in registers: none of its FP32
kernels spills a vector register, and the FP64 ones, which use all 128, spill at
most 16 (their loop's sums of statistics and a grid walk).  Read from the
kernel descriptions in the built library.  With the drain inlined the FP32
kernels spilled 18 to 322 and the FP64 ones 54 to 317, and large solves of
several cells took up to twice as long."""
import os
import re
import shutil
import subprocess

import pytest

from montecarlocpp_amd import engine

LLVM = "/opt/rocm/llvm/bin"


def kernels(tmp):
    fat, obj = os.path.join(tmp, "fat"), os.path.join(tmp, "gfx950")
    subprocess.run([f"{LLVM}/llvm-objcopy", "--dump-section", f".hip_fatbin={fat}", engine.LIB_PATH,
                    os.path.join(tmp, "rest")], check=True)
    subprocess.run([f"{LLVM}/clang-offload-bundler", "--type=o", "--unbundle", f"--input={fat}",
                    "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--output={obj}"], check=True)
    text = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", obj], check=True, capture_output=True, text=True).stdout
    out = {}
    for block in re.split(r"\n\s+- \.agpr_count", text)[1:]:
        name = re.search(r"\.symbol:\s+(\S+)", block).group(1)
        out[name] = int(re.search(r"\.vgpr_spill_count:\s+(\d+)", block).group(1))
    return out


@pytest.mark.skipif(not shutil.which(f"{LLVM}/llvm-readelf"), reason="no LLVM tools")
def test_general_kernel_does_not_spill(tmp_path):
    found = {"f": 0, "d": 0}
    for name, spills in kernels(str(tmp_path)).items():
        m = re.search(r"trajectory_kernelI([fd])", name)
        if m:
            found[m.group(1)] += 1
            assert spills <= (0 if m.group(1) == "f" else 16), (name, spills)
    assert min(found.values()) >= 12
