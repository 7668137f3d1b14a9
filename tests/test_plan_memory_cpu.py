"""Plans, their cache and device memory, on a HIP runtime without a device
(tests/native/fake_hip.cpp): what is allocated, kept and given back when
recursive levels run batched and memory is short."""
from fake_device import run


def test_low_memory_keeps_the_cache():
    """Where the batched form of recursive levels does not fit, the plan of the
    requested levels is built once and found again, and no other plan goes."""
    run("""
assert call(1024, 2, "bb", at=2) == 0 and call(1024, 1, "d", at=3) == 0
fake.fake_set_free(150 * MiB)  # batched: 1.9 GiB, as asked for 84 MiB
assert call(4096, 3, "ddd") == 0, error()
assert peak_bytes() < 100 * MiB and reported() == "DFS,DFS,DFS,"
before = count("malloc"), count("free"), count("device_sync")
for _ in range(3):
    assert call(4096, 3, "ddd") == 0, error()
    assert call(1024, 2, "bb", at=2) == 0 and call(1024, 1, "d", at=3) == 0
assert (count("malloc"), count("free"), count("device_sync")) == before
""")


def test_failed_allocation_leaves_no_error():
    """A workspace that hipMalloc refuses, whatever hipMemGetInfo said, is
    replaced by a smaller one; the refusal is not the next launch's
    error, nor the next call's after CAPS_ENOMEM."""
    run("""
fake.fake_set_malloc_limit(1 * GiB)  # batched: 1.9 GiB
assert call(4096, 3, "ddd") == 0, error()
assert peak_bytes() < 1 * GiB
assert call(8192, 2, "bb", at=2) == 3  # CAPS_ENOMEM
assert call(1024, 2, "bb", at=3) == 0, error()
import numpy as np
fake.fake_set_malloc_limit(8 * MiB)
a = np.zeros(1536 * 1536)
d = caps_amd.MatDescriptor.one_device(1536, 2, 1)
p = a.ctypes.data
assert lib.caps_multiply(p, p, p, ctypes.byref(d), None, None) == 3  # its staging
fake.fake_set_malloc_limit(1 * GiB)
assert call(512, 2, "bb", at=4) == 0, error()
fake.fake_set_malloc_limit(8)  # tables alone (no level, no workspace)
assert call(256, 0, None, at=5) != 0
fake.fake_set_malloc_limit(1 * GiB)
assert call(256, 2, "bb", at=6) == 0, error()
""")


def test_batch_plan_is_found_whatever_is_free():
    """The identical batched call finds its plan though the plan's own workspace,
    or another allocator, changed what is free."""
    run("""
for at, shapes, mode in ((1, [(2048, 2, "dd")] * 512, CRT), (2, [(1024, 2, None)] * 16, FP64),
                         (3, [(1024, 2, "bd"), (640, 1, None), (768, 1, "d")], FP64)):
    fake.fake_set_free(280 * GiB)
    assert batch(shapes, mode, at) == 0, error()
    before = count("malloc"), count("free")
    for left in (None, 200 * MiB, 0):
        if left is not None:
            fake.fake_set_free(left)
        assert batch(shapes, mode, at) == 0, error()
        assert (count("malloc"), count("free")) == before, (at, left)
fake.fake_set_free(280 * GiB)
assert batch([(1024, 2, "dd")] * 4, at=4) == 0
wide = peak_bytes()
caps_amd.set_available_memory(1)  # a budget gives the recursive plan
assert batch([(1024, 2, "dd")] * 4, at=4) == 0 and peak_bytes() < wide
""")


def test_recursive_levels_leave_memory_free():
    """Without a budget the batched form of recursive levels takes at most half
    of the free memory, and all plans' together 32 GiB more than the levels
    asked for would."""
    run("""
fake.fake_set_free(3 * GiB)
assert call(4096, 3, "ddd") == 0, error()
assert fake.fake_free() >= 3 * GiB // 2
caps_amd.release()
fake.fake_set_free(256 * GiB)
caps_amd.set_available_memory(1)
assert call(4096, 3, "ddd") == 0, error()
asked = 256 * GiB - fake.fake_free()
caps_amd.release()
caps_amd.set_available_memory(0)
assert fake.fake_free() == 256 * GiB
extra = []
for at in range(1, 25):
    assert call(4096, 3, "ddd", at=at) == 0, error()
    extra.append(256 * GiB - fake.fake_free() - at * asked)
assert max(extra) <= 32 * GiB and extra[0] > 1 * GiB, extra
assert extra[4] > 4.9 * extra[0]  # the first plans have all of theirs
""")


def test_batched_levels_keep_within_a_budget():
    """A plan is never larger than the caller's budget where the levels asked
    for fit it, whatever else a level needs (partials, exponents, alignment)."""
    run("""
for n, r, pattern, mode in ((512, 5, "ddddd", LEAF), (256, 5, "ddddd", CRT), (392, 3, "ddd", FP64),
                            (544, 5, "ddddd", CRT), (272, 4, "dddd", LEAF), (1000, 3, "dbd", CRT)):
    def peak(budget, at, entry=None):
        caps_amd.set_available_memory(budget)
        assert call(n, r, pattern, mode, at=at, entry=entry) == 0, error()
        return peak_bytes()
    for entry in (None, lib.caps_multiply_device_noalloc):
        lo, hi = peak(1, 1, entry), peak(1 << 36, 2, entry)
        assert lo < hi
        for k in range(20):
            budget = int(lo * (1.02 * hi / lo) ** (k / 19) / 8) + 1
            assert peak(budget, 3 + k, entry) <= 8 * budget, (n, r, mode, budget)
        caps_amd.release()
for count_, n, r in ((3, 256, 4), (8, 544, 5)):
    shapes = [(n, r, "d" * r)] * count_
    def peak(budget, at):
        caps_amd.set_available_memory(budget)
        assert batch(shapes, CRT, at) == 0, error()
        return peak_bytes()
    lo, hi = peak(1, 1), peak(1 << 36, 2)
    assert lo < hi
    for k in range(20):
        budget = int(lo * (1.02 * hi / lo) ** (k / 19) / 8) + 1
        assert peak(budget, 3 + k) <= 8 * budget, (n, r, budget)
    caps_amd.release()
""")


def test_plans_recorded_into_a_graph_are_kept():
    """A call on a stream under capture records its kernels, which hold the plan's
    workspace and tables: that plan goes with release() alone, the others by age
    as before."""
    run("""
S = 4096
cases = [dict(n=512, r=2, pattern="bb"), dict(n=392, r=3, pattern="dbd", bs=7, flags=8)]
caps_amd.set_available_memory(1)  # 'd' as asked: more than 16 launches
for c in cases:
    assert call(**c, stream=S) == 0, error()
shapes = [(256, 1, "b"), (320, 1, "d")]
assert batch(shapes, stream=S) == 0, error()
fake.fake_set_capturing(1)
for c in cases:
    before = count("kernel"), count("graph_launch"), count("malloc")
    assert call(**c, stream=S) == 0, error()
    assert count("kernel") > before[0]
    assert (count("graph_launch"), count("malloc")) == before[1:]
assert batch(shapes, stream=S) == 0, error()
fake.fake_set_capturing(0)
held = 256 * GiB - fake.fake_free()
for at in range(2, 62):  # 60 other plans
    assert call(256, 2, "bb", at=at) == 0, error()
mallocs = count("malloc")
for c in cases:
    assert call(**c, stream=S) == 0, error()
assert batch(shapes, stream=S) == 0 and count("malloc") == mallocs
for at in range(40, 62):  # the newest others are still there
    assert call(256, 2, "bb", at=at) == 0 and count("malloc") == mallocs
assert call(256, 2, "bb", at=2) == 0 and count("malloc") > mallocs
fake.fake_set_free(1 * MiB)  # what is short of memory takes the others only
assert call(4096, 2, "bb", at=70) == 3
mallocs = count("malloc")
assert call(**cases[0], stream=S) == 0 and count("malloc") == mallocs
caps_amd.release()
assert call(**cases[0], stream=S) == 0 and count("malloc") > mallocs
# without allocation the graph holds the host's tables
noalloc = lib.caps_multiply_device_noalloc
fake.fake_copy_src.restype = ctypes.c_void_p
fake.fake_set_capturing(1)
assert call(512, 4, "dddd", stream=S, entry=noalloc) == 0, error()
n = ctypes.c_size_t()
src = fake.fake_copy_src(ctypes.byref(n))
tables = ctypes.string_at(src, n.value)
fake.fake_set_capturing(0)
for at in range(2, 40):
    assert call(512, 4, "dddd", at=at, stream=S, entry=noalloc) == 0, error()
assert ctypes.string_at(src, n.value) == tables
""")
