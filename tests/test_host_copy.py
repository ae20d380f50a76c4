"""csrc/fr_host_copy.cpp against a model of the HIP runtime (host_copy_model.cpp): copies between host
arrays and the device come after the work queued on the caller's stream, whatever stream that is, and
arrays that the runtime knows are not copied twice."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.join(os.path.dirname(HERE), "fluxreconstruction.jl_amd")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_copies_against_the_model(tmp_path):
    exe, objs = str(tmp_path / "model"), []
    for src in (os.path.join(HERE, "host_copy_model.cpp"), os.path.join(PKG, "csrc", "fr_host_copy.cpp")):
        objs.append(str(tmp_path / (os.path.basename(src) + ".o")))
        subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", "-O1", "-fPIC", "-I", os.path.join(PKG, "csrc"),
                        "-c", src, "-o", objs[-1]], check=True)
    subprocess.run(["g++", *objs, "-o", exe, "-pthread"], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout
