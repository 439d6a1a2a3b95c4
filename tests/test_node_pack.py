"""The packed BVH4 node (no GPU): its boxes contain the float boxes, and its
slab test passes every box that the float slab test passes
(tests/pack_check.cpp)."""
import os
import subprocess

from colvillea_amd import build as hipbuild

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_packed_nodes_cull_nothing_more(tmp_path):
    exe = str(tmp_path / "pack_check")
    src = os.path.join(REPO, "tests", "pack_check.cpp")
    subprocess.run([hipbuild.hipcc(), "-std=c++17", "-O2", "-ffp-contract=off", "-fno-gpu-rdc", src, "-o", exe],
                   check=True, capture_output=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout
