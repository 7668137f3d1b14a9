"""FP64 leaf GEMM where the tiles do not divide over the CUs: the ones left over
run as four tiles of half the size.  Counts of products that leave from a few
tiles to almost one per CU, whole and ragged sizes: every product has the bits
of the product alone (all tiles sum in the same K order), which
test_gpu_leaf_tiles checks against NumPy."""
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


@pytest.mark.parametrize("m", [48, 64, 65, 128, 130, 200, 256, 321])
@pytest.mark.parametrize("count", [49, 65, 137, 261, 343])
def test_left_over_tiles_give_the_same_bits(m, count):
    print(f"[gpu] m={m} count={count}", flush=True)
    rng = np.random.default_rng(m)
    A, B = (torch.from_numpy(x).cuda() for x in rng.uniform(-1, 1, (2, m * m)))
    d = caps_amd.MatDescriptor.one_device(m, 0, 1)
    C = torch.full_like(A, float("nan"))
    caps_amd.multiply_device(A, B, C, d, "")
    out = torch.full((count, m * m), float("nan"), dtype=torch.float64, device="cuda")
    caps_amd.multiply_batch_device([A] * count, [B] * count, list(out), [d] * count, [""] * count)
    torch.cuda.synchronize()
    assert torch.equal(out, C.expand(count, m * m))
    caps_amd.release()
