"""Scale exponents of the residue modes: every entry of a row of A and of a
column of B counts.  One entry per row (column) is far larger than the rest, at
a random place, so an entry that no partial reads gives wrong exponents and
other bits than the exact model's (oracle/split.py).  Orders at the edges of the
64-row blocks, of the 4 waves' shares of a chunk and of the 8-column steps."""
import numpy as np
import pytest

import caps_amd
import oracle
from oracle import split

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _setup():
    oracle.build()
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    caps_amd.load()
    yield
    caps_amd.release()


@pytest.mark.parametrize("m,r,bs", [(1, 1, 1), (3, 2, 1), (5, 1, 5), (31, 1, 1), (32, 1, 8), (33, 1, 1),
                                    (64, 0, 1), (65, 1, 13), (127, 1, 1), (129, 1, 3), (257, 1, 1)])
def test_every_entry_counts(m, r, bs):
    n = m << r
    rng = np.random.default_rng(100 * m + r)
    A, B = rng.uniform(-1, 1, (2, n, n))
    where = rng.integers(0, n, (2, n))
    A[np.arange(n), where[0]] *= 2.0 ** 12
    B[where[1], np.arange(n)] *= 2.0 ** 12
    A[n // 2] = 0.0
    print(f"[gpu] n={n} r={r} bs={bs}", flush=True)
    d = caps_amd.MatDescriptor.one_device(n, r, bs)
    a, b = (torch.from_numpy(oracle.to_caps(x, r, bs)).cuda() for x in (A, B))
    c = torch.full_like(a, float("nan"))
    caps_amd.multiply_device(a, b, c, d, "b" * r, mode=caps_amd.MODE_CRT_INT8)
    torch.cuda.synchronize()
    assert np.array_equal(oracle.from_caps(c.cpu().numpy(), n, r, bs), split.crt_mode(A, B, 14))
