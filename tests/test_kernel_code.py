"""What the compiler made of the 2D stage and residual kernels, read from the built library's own code."""
import glob
import os
import re
import shutil
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fluxreconstruction.jl_amd", "frhip",
                   "libfrhip.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.mark.skipif(not (os.path.exists(LIB) and os.path.exists(OBJDUMP)), reason="needs the library and llvm-objdump")
def test_buffer_accesses_take_their_plane_from_scalars(tmp_path):
    """The plane offset of a buffer access is uniform over a wavefront.  Where the compiler loses sight of
    that it wraps the access in a loop over the lanes' values (readfirstlane .. xor exec, branch back)."""
    lib = shutil.copy(LIB, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True)
    seen, loops = 0, {}
    for image in glob.glob(lib + ".*gfx950"):
        with open(image, "rb") as f:
            if b"fr2d_kernel" not in f.read():
                continue
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", image], check=True,
                              capture_output=True, text=True).stdout
        for name, body in re.findall(r"<(\S*fr2d_kernel\S*)>:\n(.*?)(?=\n\n|\Z)", text, re.S):
            seen += 1
            n = len(re.findall(r"s_xor_b64 exec,.*\n(?:.*\n)?\s*s_cbranch_execnz", body))
            if n:
                loops[name] = n
    assert seen > 100 and not loops, loops
