"""Errors of the host-array calls, on a HIP runtime without a device: a call that
fails returns with nothing still reading the pinned ring or the caller's arrays."""
from fake_device import run


def test_failed_layout_conversion_settles_its_copies():
    run("""
import numpy as np
a, b = np.zeros((2, 1024 * 1024))
d = caps_amd.MatDescriptor.one_device(1024, 2, 8)
for f in (lib.caps_to_layout, lib.caps_from_layout):
    assert f(a.ctypes.data, b.ctypes.data, ctypes.byref(d)) == 0, error()
fake.fake_fail_launch(b"kernel")
for f in (lib.caps_to_layout, lib.caps_from_layout):
    before = count("stream_sync")
    assert f(a.ctypes.data, b.ctypes.data, ctypes.byref(d)) == 4, error()  # CAPS_EHIP
    assert count("stream_sync") > before
    before = count("stream_sync")
    assert lib.caps_multiply(a.ctypes.data, a.ctypes.data, b.ctypes.data, ctypes.byref(d), None,
                             None) == 4
    assert count("stream_sync") > before
""")
