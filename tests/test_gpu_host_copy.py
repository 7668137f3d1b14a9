"""Host arrays in and out: the bits of the device call, at matrices below, at
and past one 2 MiB chunk, past the ring of eight, with a ragged last piece; from
pageable and pinned memory, unaligned arrays, A as B and as C, several threads
at a time, and after a release."""
import ctypes
import threading

import numpy as np
import pytest

import caps_amd

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _setup():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    caps_amd.load()
    yield
    caps_amd.release()


def _device(A, B, d):
    a, b = torch.from_numpy(A.copy()).cuda(), torch.from_numpy(B.copy()).cuda()
    c = torch.empty_like(a)
    caps_amd.multiply_device(a, b, c, d)
    torch.cuda.synchronize()
    return c.cpu().numpy()


@pytest.mark.parametrize("n", [1, 8, 256, 511, 512, 513, 724, 1026, 1450, 2304])
def test_host_call_gives_the_device_bits(n):
    print(f"[gpu] n={n}", flush=True)
    r = 1 if n % 2 == 0 else 0
    d = caps_amd.MatDescriptor.one_device(n, r, 1)
    A, B = np.random.default_rng(n).uniform(-1, 1, (2, n * n))
    want = _device(A, B, d)
    for _ in range(2):
        C = np.full(n * n, np.nan)
        caps_amd.multiply(A, B, C, d)
        assert np.array_equal(C, want)
    # 8-byte aligned arrays
    a, b, c = (np.empty(n * n + 1)[1:] for _ in range(3))
    a[:], b[:] = A, B
    caps_amd.multiply(a, b, c, d)
    assert np.array_equal(c, want)
    # pinned A and C beside a pageable B
    pa, pc = (torch.empty(n * n, dtype=torch.float64, pin_memory=True).numpy() for _ in range(2))
    pa[:] = A
    caps_amd.multiply(pa, B, pc, d)
    assert np.array_equal(pc, want)


def test_the_result_over_an_operand_and_a_square():
    n = 700
    d = caps_amd.MatDescriptor.one_device(n, 2, 1)
    A, B = np.random.default_rng(1).uniform(-1, 1, (2, n * n))
    want, square = _device(A, B, d), _device(A, A, d)
    C = A.copy()
    caps_amd.multiply(C, B, C, d)
    assert np.array_equal(C, want)
    caps_amd.multiply(A, A, C, d)
    assert np.array_equal(C, square)


def test_several_threads_and_a_release_between():
    sizes = [300, 640, 1100, 1600]
    data = [(n, caps_amd.MatDescriptor.one_device(n, 2, 1),
             *np.random.default_rng(n).uniform(-1, 1, (2, n * n))) for n in sizes]
    want = [_device(A, B, d) for _, d, A, B in data]
    for _ in range(2):
        out = [np.full(n * n, np.nan) for n in sizes]

        def work(i):
            for _ in range(3):
                caps_amd.multiply(data[i][2], data[i][3], out[i], data[i][1])

        threads = [threading.Thread(target=work, args=(i,)) for i in range(len(sizes))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        for o, w in zip(out, want):
            assert np.array_equal(o, w)
        caps_amd.release()


@pytest.mark.parametrize("n,bs", [(56, 7), (600, 5), (1536, 8)])
def test_layout_of_host_arrays_round_trips(n, bs):
    d = caps_amd.MatDescriptor.one_device(n, 2, bs)
    X = np.random.default_rng(n).uniform(-1, 1, n * n)
    caps, back = np.full(n * n, np.nan), np.full(n * n, np.nan)
    lib = caps_amd.load()

    def host(entry, src, dst):  # the C entry points: the Python module wraps the device ones
        entry.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.POINTER(caps_amd.MatDescriptor)]
        assert entry(src.ctypes.data, dst.ctypes.data, ctypes.byref(d)) == 0

    host(lib.caps_to_layout, X, caps)
    t = torch.from_numpy(X).cuda()
    dev = torch.empty_like(t)
    caps_amd.to_layout_device(t, dev, d)
    assert np.array_equal(caps, dev.cpu().numpy())
    host(lib.caps_from_layout, caps, back)
    assert np.array_equal(back, X)
