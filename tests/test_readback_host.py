"""A reading that fails after its kernels were queued must not give its pinned
block back while they may still write it.  readback.hip is compiled for the
host and linked with stubs of the HIP runtime (no GPU needed)."""
import os
import re
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "freeflow_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def run(cmd):
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0, r.stdout
    return r.stdout


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_blocks_are_lent_again_only_after_a_wait(tmp_path):
    obj, stub, exe = (str(tmp_path / n) for n in ("readback.o", "stub.o", "check"))
    flags = ["--offload-arch=gfx950", "--offload-host-only", "-std=c++17", "-fPIC", "-Xclang", "-target-feature",
             "-Xclang", "-packed-fp32-ops"]
    run([HIPCC, *flags, "-O1", "-c", os.path.join(CSRC, "readback.hip"), "-o", obj])
    run([HIPCC, *flags, "-x", "hip", "-c", os.path.join(HERE, "native", "readback_wait_check.cpp"), "-o", stub])
    fatbins = set(re.findall(r"__hip_fatbin_[0-9a-f]+", run(["nm", obj]) + run(["nm", stub])))
    defs = [f"-Wl,--defsym={f}=__hip_fatbin_stub" for f in fatbins]
    run(["g++", "-o", exe, obj, stub, *defs, "-lpthread"])
    out = run([exe])
    print(out)
    assert "wrong 0" in out
