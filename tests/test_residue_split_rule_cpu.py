"""A's residue split is fused with its two top levels where the whole multiply
measured faster so (the figures at bb_split_a_pays in fused2.hip)."""
from fake_device import run


def test_fused_where_it_measured_faster():
    run("""
for n, fused in ((512, 0), (1024, 0), (2048, 0), (2560, 1), (3072, 0), (3584, 1), (4096, 1),
                 (4608, 1), (5120, 1), (5632, 1)):
    before = count("bb_split_a_kernel"), count("crt_split_a_kernel")
    assert call(n, 2, "bb", CRT) == 0, error()
    after = count("bb_split_a_kernel"), count("crt_split_a_kernel")
    assert (after[0] - before[0], after[1] - before[1]) == (fused, 1 - fused), n
""")
