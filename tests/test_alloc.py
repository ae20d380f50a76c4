"""The library's host code, compiled for the host alone, on a stand-in of the HIP runtime (alloc_model.cpp): host
allocations that fail inside the create calls, one after another (FR_E_NOMEM, no exception), captures that
are kept, launch sizes."""
import os
import subprocess

import pytest

from test_host_copy import HERE, HIPCC, PKG


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_no_exception_leaves_the_create_calls(tmp_path):
    exe, objs = str(tmp_path / "model"), []
    csrc = os.path.join(PKG, "csrc")
    for src in [os.path.join(HERE, "alloc_model.cpp")] + [os.path.join(csrc, f) for f in (
            "fr1d.hip", "fr2d_api.hip", "fr_bgk.hip", "fr_bgk1d.hip", "fr_host_copy.cpp", "fr_host_ops.cpp")]:
        objs.append(str(tmp_path / (os.path.basename(src) + ".o")))
        subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", "-O1", "-fPIC", "-Wno-unused-result",
                        "-I", csrc, "-c", src, "-o", objs[-1]], check=True)
    # the device code that the objects name is not there, and the stand-in does not look at it; nor are the
    # launches of 2D steps, which are not called
    subprocess.run(["g++", *objs, "-o", exe, "-pthread", "-Wl,--unresolved-symbols=ignore-all"], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, (out.returncode, out.stdout, out.stderr)
