"""Residue leaves at a 16-byte pitch: orders that are not a multiple of 16, at
the edges of a 16-byte chunk, of the 32 x 128 split tile and of the 128 and
256 block tiles, in INT8 and BF16 and the leaf-only split, plain and blocked
leaves, batched and recursive levels.

The residue modes return the correctly rounded product of the truncated
operands whatever the pattern, so every route gives the bits of the exact
model (oracle/split.py)."""
import numpy as np
import pytest

import caps_amd
import oracle
from oracle import split

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

INT8, BF16, LEAF = caps_amd.MODE_CRT_INT8, caps_amd.MODE_CRT_BF16, caps_amd.MODE_OZAKI_INT8


@pytest.fixture(scope="module", autouse=True)
def _setup():
    oracle.build()
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    caps_amd.load()
    yield
    caps_amd.release()


def _data(n):
    rng = np.random.default_rng(n)
    e = np.ldexp(1.0, rng.integers(-10, 11, (2, n, n)))
    return rng.uniform(-1, 1, (2, n, n)) * e


def _run(A, B, n, r, bs, pattern, mode, entry=caps_amd.multiply_device):
    print(f"[gpu] n={n} r={r} bs={bs} {pattern} mode={mode}", flush=True)
    d = caps_amd.MatDescriptor.one_device(n, r, bs)
    a, b = (torch.from_numpy(oracle.to_caps(x, r, bs)).cuda() for x in (A, B))
    c = torch.full_like(a, float("nan"))
    entry(a, b, c, d, pattern, mode=mode)
    torch.cuda.synchronize()
    return oracle.from_caps(c.cpu().numpy(), n, r, bs)


@pytest.mark.parametrize("m,r,bs,patterns", [
    (1, 2, 1, ["bb", "bd"]), (3, 3, 1, ["bbd"]), (15, 2, 1, ["bb", "dd"]), (17, 2, 17, ["bb"]),
    (31, 2, 1, ["bb", "db"]), (33, 1, 11, ["b", "d"]), (50, 2, 5, ["bb", "bd"]),
    (63, 2, 1, ["bb"]), (65, 1, 1, ["b"]), (97, 2, 1, ["bb", "bd"]), (127, 1, 1, ["b"]),
    (130, 2, 1, ["bb"]), (257, 1, 1, ["b"])])
def test_ragged_leaves_give_the_model_bits(m, r, bs, patterns):
    n = m << r
    A, B = _data(n)
    want = split.crt_mode(A, B, 14)
    for p in patterns:
        for mode in (INT8, BF16):
            assert np.array_equal(_run(A, B, n, r, bs, p, mode), want), (p, mode)
        assert np.array_equal(_run(A, B, n, r, bs, p, INT8, caps_amd.multiply_device_noalloc), want)


@pytest.mark.parametrize("m", [515, 750, 1001])
def test_ragged_large_leaves_agree(m):
    """Past the model's reach: the 256-tile kernel with partial edges, the
    128-tile kernel and BF16 give the same bits, batched or recursive."""
    n = 2 * m
    A, B = _data(n)
    want = _run(A, B, n, 1, 1, "b", INT8)
    scale = np.abs(A) @ np.abs(B)
    assert (np.abs(want - A @ B) <= 4 * n * 2.0 ** -53 * scale).all()
    small = lambda *a, **k: caps_amd.multiply_device(*a, flags=caps_amd.FLAG_SMALL_TILE, **k)
    assert np.array_equal(_run(A, B, n, 1, 1, "b", INT8, small), want)
    assert np.array_equal(_run(A, B, n, 1, 1, "d", INT8), want)
    assert np.array_equal(_run(A, B, n, 1, 1, "b", BF16), want)


@pytest.mark.parametrize("m", [50, 64, 90, 96, 97, 126, 128, 150, 160, 161, 300, 320, 380, 384,
                               570, 576, 640])
def test_int8_tiles_equal_bf16(m):
    """686 INT8 products on each of the block tiles 64, 96, 128, 160, 192 and
    256, whole and partial, give the bits of the BF16 kernels (another tile,
    another accumulation)."""
    n = 4 * m
    g = torch.Generator(device="cuda")
    g.manual_seed(m)
    A, B = torch.rand((2, n * n), generator=g, device="cuda", dtype=torch.float64) * 2 - 1
    d = caps_amd.MatDescriptor.one_device(n, 2, 1)
    out = []
    for mode, flags in ((BF16, 0), (INT8, 0), (INT8, caps_amd.FLAG_SMALL_TILE)):
        print(f"[gpu] n={n} bb mode={mode} flags={flags}", flush=True)
        C = torch.full_like(A, float("nan"))
        caps_amd.multiply_device(A, B, C, d, "bb", mode=mode, flags=flags)
        torch.cuda.synchronize()
        out.append(C)
    assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])
    caps_amd.release()


@pytest.mark.parametrize("m", [1, 15, 18, 49, 66])
def test_leaf_split_ragged(m):
    n = 2 * m
    A, B = _data(n)
    want = split.leaf_split_mode(A, B, 1, 14)
    assert np.array_equal(_run(A, B, n, 1, 1, "b", LEAF), want)


@pytest.mark.parametrize("n,r,pattern", [(320, 6, "bbbbbb"), (576, 6, "bbbbdd"),
                                         (608, 5, "bbbbd"), (1152, 5, "dbbbb"),
                                         (1504, 5, "bdddb"), (2284, 2, "dd")])
def test_noalloc_keeps_what_fitted_without_the_pitch(n, r, pattern):
    """Plans that are close to the scratch limit without the pitch, and pass it
    with it (leaves of 5 -> 16, 9 -> 16, 19 -> 32 ...), still run, with the same
    bits; one that is over the limit without it is refused as before."""
    A, B = _data(n)
    want = _run(A, B, n, r, 1, pattern, INT8)
    got = _run(A, B, n, r, 1, pattern, INT8, caps_amd.multiply_device_noalloc)
    assert np.array_equal(got, want)
    caps_amd.release()


def test_noalloc_limit_does_not_count_the_pitch():
    n, r = 2308, 2  # 14 (3 + 2/4 + 2/16) n^2 bytes = 257.8 MiB
    A, B = _data(n)
    with pytest.raises(caps_amd.CapsError) as e:
        _run(A, B, n, r, 1, "dd", INT8, caps_amd.multiply_device_noalloc)
    assert e.value.code == 3
