"""Copies between device memory and the caller's buffers (no GPU): what
HostCopier does with the runtime's calls, against a stand-in for them
(tests/host_copy_check.cpp)."""
import os
import subprocess

import pytest

from colvillea_amd import build as hipbuild

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("host_copy") / "host_copy_check")
    include = os.path.join(os.path.dirname(os.path.dirname(os.path.realpath(hipbuild.hipcc()))), "include")
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", include, "-pthread",
                    os.path.join(REPO, "tests", "host_copy_check.cpp"),
                    os.path.join(REPO, "colvillea_amd", "csrc", "host_copy.cpp"), "-o", out], check=True, capture_output=True)
    return out


# sizes: every size arrives whole, up and down
# no_pinned: without pinned memory copies still work
# pinned: the caller's own pinned memory takes one copy, not two
# wait: behind a render still running only the calling thread waits
# setup: tiny readbacks make 16 KiB of pinned memory, once there are several; small copies none, large ones a bounded staging
# device: where another device than the context's is current, as it would be without staging
@pytest.mark.parametrize("case", ["sizes", "no_pinned", "pinned", "wait", "setup", "device"])
def test_copies(exe, case):
    r = subprocess.run([exe, case], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
