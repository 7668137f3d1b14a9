"""FP64 leaf GEMM on its three block tiles (128, 64, 32), at the sizes where a
tile, a K slice of 16 or a 16-byte chunk is partial.

One product alone takes the smallest tile, CAPS_FLAG_SMALL_TILE the 64 tile,
and a batch that fills the device the 128 tile where its padding is small.
Every tile sums each element's products in the same K order, so all three give
the same bits; they are checked against NumPy within 2 m u (|A||B|) per
element (m products and m sums, each rounded once, on either side)."""
import numpy as np
import pytest

import caps_amd

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

U = 2.0 ** -53


@pytest.fixture(scope="module", autouse=True)
def _setup():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    caps_amd.load()
    yield
    caps_amd.release()


def _single(A, B, m, flags=0):
    """C (column-major) = A B, one leaf of order m; C starts as NaN with NaN
    around it, which must stay."""
    pad = torch.full((m * m + 64,), float("nan"), dtype=torch.float64, device="cuda")
    C = pad[32:32 + m * m]
    caps_amd.multiply_device(A, B, C, caps_amd.MatDescriptor.one_device(m, 0, 1), "", flags=flags)
    torch.cuda.synchronize()
    assert torch.isnan(pad[:32]).all() and torch.isnan(pad[32 + m * m:]).all()
    return C.clone()


@pytest.mark.parametrize("m", [1, 2, 3, 15, 16, 17, 18, 31, 32, 33, 49, 63, 64, 65, 66, 96, 113,
                               127, 128, 129, 144, 250, 255, 256, 257, 375, 625])
def test_tiles_agree_and_match(m):
    print(f"[gpu] leaf m={m}", flush=True)
    rng = np.random.default_rng(m)
    a, b = rng.uniform(-1, 1, (2, m, m))
    A = torch.from_numpy(np.asfortranarray(a).ravel(order="F").copy()).cuda()
    B = torch.from_numpy(np.asfortranarray(b).ravel(order="F").copy()).cuda()
    C = _single(A, B, m)
    got = C.cpu().numpy().reshape((m, m), order="F")
    assert (np.abs(got - a @ b) <= 4 * m * U * (np.abs(a) @ np.abs(b))).all()
    assert torch.equal(C, _single(A, B, m, caps_amd.FLAG_SMALL_TILE))
    count = 512  # fills the device: the tile with the least padding
    out = torch.full((count, m * m), float("nan"), dtype=torch.float64, device="cuda")
    d = caps_amd.MatDescriptor.one_device(m, 0, 1)
    caps_amd.multiply_batch_device([A] * count, [B] * count, list(out), [d] * count, [""] * count)
    torch.cuda.synchronize()
    assert torch.equal(out, C.expand(count, m * m))
    caps_amd.release()


@pytest.mark.parametrize("m", [31, 49, 50, 130])
def test_infinities_stay_in_their_row_and_column(m):
    """Rows, columns and k beyond m are zeros or discarded, never read into an
    element they do not belong to."""
    print(f"[gpu] infinities m={m}", flush=True)
    rng = np.random.default_rng(m)
    a, b = rng.uniform(0.5, 1, (2, m, m))
    a[0, m - 1] = np.inf   # read as the row after the last by a tile that runs over
    b[0, m // 2] = np.inf  # first k of a column: the k after the last of the one before
    A = torch.from_numpy(a.ravel(order="F").copy()).cuda()
    B = torch.from_numpy(b.ravel(order="F").copy()).cuda()
    want = np.zeros((m, m), bool)
    want[0, :] = True
    want[:, m // 2] = True
    for flags in (0, caps_amd.FLAG_SMALL_TILE):
        got = _single(A, B, m, flags).cpu().numpy().reshape((m, m), order="F")
        assert (np.isinf(got) == want).all() and not np.isnan(got).any()
    caps_amd.release()
