"""What the tests of the contraction kernels share."""
import os
import re
import subprocess

from akg_amd import driver


def compiled_notes(text, folder):
    """The kernel of a description compiled into the (empty) folder `folder`, and of its code the scratch a lane and the registers."""
    kernel = driver.HipKernel(text, out_dir=str(folder))
    notes = "".join(subprocess.run(["/opt/rocm/llvm/bin/llvm-readelf", "--notes", str(f)], capture_output=True, text=True, check=True).stdout
                    for f in folder.glob("*.hsaco"))
    scratch = max(int(x) for x in re.findall(r"\.private_segment_fixed_size:\s+(\d+)", notes))
    registers = max(int(x) for x in re.findall(r"\.vgpr_count:\s+(\d+)", notes))
    return kernel, scratch, registers


def disassembled(text, folder):
    """... and its code."""
    kernel = driver.HipKernel(text, out_dir=str(folder))
    objdump = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")
    return kernel, "".join(subprocess.run([objdump, "-d", str(f)], check=True, capture_output=True, text=True).stdout for f in folder.glob("*.hsaco"))
