"""Merged launches of a batch and interleaved C segments
(tests/native/merge_segments_check.cpp)."""
import os
import subprocess

import caps_amd
from fake_device import ROOT


def test_products_with_segments_are_not_merged(tmp_path):
    exe = tmp_path / "merge_segments_check"
    lib = os.path.dirname(caps_amd.LIB_PATH)
    r = subprocess.run(["/opt/rocm/bin/hipcc", "-O1", "-std=c++17", "-x", "hip",
                        "--offload-arch=gfx950", "-I", os.path.join(ROOT, "include"),
                        os.path.join(ROOT, "tests", "native", "merge_segments_check.cpp"),
                        "-o", str(exe), "-L", lib, "-lcaps_amd", f"-Wl,-rpath,{lib}"],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout == "OK\n", r.stdout + r.stderr
