"""The fused passes' plans take every pass the schedules make (no GPU).

orth_host.cpp is compiled with g++ against the host-only HIP stand-in
(tests/host_harness), with the plan functions of the built library in place of
the stand-in's; tests/host_harness/plans.cpp then enqueues every variant for
every column count up to 530 at block widths 1 to 32 (device form, fixed
scratch, FP32 storage with FP64 products).  A schedule that runs fused for a
size some pass of which its plan refuses would fail part-way, with X already
overwritten.
"""
import os
import shutil
import subprocess

import pytest

import bcgs_hip as B

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(ROOT, "one-synchronization-bcgs_amd", "csrc")
HARNESS = os.path.join(HERE, "host_harness")


def test_every_pass_of_every_schedule_has_a_plan(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    inc = ["-std=c++17", "-O1", "-I" + HARNESS, "-I" + CSRC, "-I" + os.path.join(ROOT, "include")]
    # The stand-in's own plans step aside under other names.
    names = ["pass_rows", "pass_wg_per_cu", "launch_pass"]
    rename = ["-D%s=stub_%s" % (n, n) for n in names]
    src = open(os.path.join(CSRC, "orth_host.cpp")).read()
    src = src.replace('"../../include/orth.h"', '"orth.h"')
    src = src.replace('"../../include/orth_ext.h"', '"orth_ext.h"')
    host = tmp_path / "orth_host.cpp"
    host.write_text(src)
    objs = []
    for name, path, extra in [("host", str(host), []),
                              ("stub", os.path.join(HARNESS, "hip_stub.cpp"), rename),
                              ("plans", os.path.join(HARNESS, "plans.cpp"), [])]:
        obj = str(tmp_path / (name + ".o"))
        r = subprocess.run(["g++"] + inc + extra + ["-c", path, "-o", obj], capture_output=True,
                           text=True, timeout=600)
        assert r.returncode == 0, r.stderr[-4000:]
        objs.append(obj)
    exe = str(tmp_path / "plans")
    r = subprocess.run(["g++"] + objs + ["-o", exe, "-lpthread", "-ldl"], capture_output=True,
                       text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([exe, B.LIB_PATH], capture_output=True, text=True, timeout=900)
    assert r.returncode == 0, (r.stdout + r.stderr)[-4000:]
    assert "refused 0" in r.stdout
