"""The limit of caps_multiply_device_noalloc (CAPS_NOALLOC_SCRATCH_MIB of tables
and workspace, without the padding of residue leaves), on a HIP runtime without a
device: calls close to it run, calls over it are refused."""
import os
import subprocess

import caps_amd
from fake_device import ROOT, run

NOALLOC = """
def noalloc(n, r, pattern, mode, moduli=14):
    return call(n, r, pattern, mode, moduli=moduli, entry=lib.caps_multiply_device_noalloc)
"""


def test_leaf_split_is_counted_without_the_pitch():
    run(NOALLOC + """
for n, r, pattern in ((4272, 1, "d"), (4294, 1, "d"), (5928, 2, "dd"), (1606, 1, "b")):
    assert noalloc(n, r, pattern, LEAF) == 0, (n, error())
for n, r, pattern in ((4302, 1, "d"), (1610, 1, "b")):
    assert noalloc(n, r, pattern, LEAF) == 3, n
""")


def test_padded_plans_that_fitted_without_the_pitch():
    """Leaves of 17, 33 and 34 (pitch 32 and 48) at 6 and 7 levels, where the
    tables take a third of the limit: all ran before the leaves had a pitch."""
    run(NOALLOC + """
for pattern, k in (("dddddbb", 8), ("dbdddbb", 6), ("bddbddb", 3), ("dbdbbbb", 3)):
    assert noalloc(2176, 7, pattern, CRT, k) == 0, (pattern, error())
    assert reported() == "".join("BFS," if p == "b" else "DFS," for p in pattern)
assert noalloc(2176, 7, "dddddbb", CRT, 9) == 3
for n, r, pattern, k in ((2176, 6, "ddddbb", 14), (2176, 6, "dddddb", 14), (2112, 6, "dddbdb", 14),
                         (2112, 5, "ddddb", 16)):
    assert noalloc(n, r, pattern, CRT, k) == 0, (n, pattern, error())
""")


def test_tables_in_parts(tmp_path):
    """tests/native/table_parts_check.cpp against the built library."""
    exe = tmp_path / "table_parts_check"
    lib = os.path.dirname(caps_amd.LIB_PATH)
    r = subprocess.run(["/opt/rocm/bin/hipcc", "-O1", "-std=c++17", "-x", "hip",
                        "--offload-arch=gfx950", "-I", os.path.join(ROOT, "include"),
                        os.path.join(ROOT, "tests", "native", "table_parts_check.cpp"),
                        "-o", str(exe), "-L", lib, "-lcaps_amd", f"-Wl,-rpath,{lib}"],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout == "OK\n", r.stdout + r.stderr
