"""The limit of caps_multiply_device_noalloc (CAPS_NOALLOC_SCRATCH_MIB of tables
and workspace, without the padding of residue leaves), on a HIP runtime without a
device: calls close to it run, calls over it are refused."""
from fake_device import run

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
