"""A's residue split with leaves that are multiples of 128, on both sides of the
rule that fuses it with its two top levels: the bits of the level-by-level run
(FLAG_NO_FUSION; the residue modes are exact, so every route gives the same)."""
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


@pytest.mark.parametrize("n,pattern,bs,mode", [
    (512, "bb", 1, caps_amd.MODE_CRT_INT8), (1024, "bbb", 1, caps_amd.MODE_CRT_BF16),
    (2048, "bb", 512, caps_amd.MODE_CRT_INT8), (2560, "bb", 1, caps_amd.MODE_CRT_INT8),
    (2560, "bb", 640, caps_amd.MODE_CRT_BF16), (3072, "bb", 1, caps_amd.MODE_CRT_INT8),
    (4096, "bbb", 1, caps_amd.MODE_CRT_INT8)])
def test_bits_on_both_sides(n, pattern, bs, mode):
    print(f"[gpu] n={n} {pattern} bs={bs} mode={mode}", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    A, B = torch.rand((2, n * n), generator=g, device="cuda", dtype=torch.float64) * 2 - 1
    d = caps_amd.MatDescriptor.one_device(n, len(pattern), bs)
    out = []
    for flags in (0, caps_amd.FLAG_NO_FUSION):
        C = torch.full_like(A, float("nan"))
        caps_amd.multiply_device(A, B, C, d, pattern, mode=mode, flags=flags)
        torch.cuda.synchronize()
        out.append(C)
        caps_amd.release()
    assert not torch.isnan(out[0]).any()
    assert torch.equal(out[0], out[1])
