"""Which memory the end of a call writes to from a kernel, and which through
copies (no GPU): orth_host.cpp against the host-only HIP stand-in, with the
pointer attributes, the strided copy and the small steps of
tests/host_harness/result_copy.cpp.
"""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(ROOT, "one-synchronization-bcgs_amd", "csrc")
HARNESS = os.path.join(HERE, "host_harness")


def test_kernels_write_only_what_they_can_address(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    inc = ["-std=c++17", "-O1", "-I" + HARNESS, "-I" + CSRC, "-I" + os.path.join(ROOT, "include")]
    rename = ["-D%s=stub_%s" % (n, n)
              for n in ("hipPointerGetAttributes", "hipMemcpy2DAsync", "launch_small")]
    src = open(os.path.join(CSRC, "orth_host.cpp")).read()
    src = src.replace('"../../include/orth.h"', '"orth.h"')
    src = src.replace('"../../include/orth_ext.h"', '"orth_ext.h"')
    host = tmp_path / "orth_host.cpp"
    host.write_text(src)
    objs = []
    for name, path, extra in [("host", str(host), []),
                              ("stub", os.path.join(HARNESS, "hip_stub.cpp"), rename),
                              ("copy", os.path.join(HARNESS, "result_copy.cpp"), [])]:
        obj = str(tmp_path / (name + ".o"))
        r = subprocess.run(["g++"] + inc + extra + ["-c", path, "-o", obj], capture_output=True,
                           text=True, timeout=600)
        assert r.returncode == 0, r.stderr[-4000:]
        objs.append(obj)
    exe = str(tmp_path / "copy")
    r = subprocess.run(["g++"] + objs + ["-o", exe, "-lpthread"], capture_output=True, text=True,
                       timeout=600)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
