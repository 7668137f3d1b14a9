"""Plans, their cache and device memory, on a HIP runtime without a device
(tests/native/fake_hip.cpp): what is allocated, kept and given back when
recursive levels run batched and memory is short."""
from fake_device import run


def test_low_memory_keeps_the_cache():
    """Where the batched form of recursive levels does not fit, the plan of the
    requested levels is built once and found again, and no other plan goes."""
    run("""
assert call(1024, 2, "bb", at=2) == 0 and call(1024, 1, "d", at=3) == 0
fake.fake_set_free(1 * GiB)  # batched: 1.9 GiB
assert call(4096, 3, "ddd") == 0, error()
assert peak_bytes() < 100 * MiB and reported() == "DFS,DFS,DFS,"
before = count("malloc"), count("free"), count("device_sync")
for _ in range(3):
    assert call(4096, 3, "ddd") == 0, error()
    assert call(1024, 2, "bb", at=2) == 0 and call(1024, 1, "d", at=3) == 0
assert (count("malloc"), count("free"), count("device_sync")) == before
""")
