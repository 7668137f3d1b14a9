"""Recursive ('d') levels that run batched because their workspace is small:
the reported pattern is the requested one, a memory budget keeps the levels
recursive, and the bits are the same either way (BFS and DFS steps evaluate
the same expression trees)."""
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
    caps_amd.set_available_memory(0)
    caps_amd.release()


@pytest.mark.parametrize("mode", [caps_amd.MODE_FP64, caps_amd.MODE_OZAKI_INT8,
                                  caps_amd.MODE_CRT_INT8])
@pytest.mark.parametrize("n,r,bs,pattern,cutoff", [
    (392, 3, 7, "ddd", 0), (392, 3, 7, "bdd", 0), (392, 3, 7, "dbd", 0), (384, 2, 1, "dh", 0),
    (64, 6, 1, "dddddd", 0), (1024, 3, 1, "ddb", 0), (1024, 3, 1, "ddd", 1)])
def test_small_recursive_levels(n, r, bs, pattern, cutoff, mode):
    if cutoff and mode == caps_amd.MODE_OZAKI_INT8:
        pytest.skip("the leaf-only split has no cutoff")
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    A, B = torch.rand((2, n * n), generator=g, device="cuda", dtype=torch.float64) * 2 - 1
    d = caps_amd.MatDescriptor.one_device(n, r, bs)
    out, peak = [], []
    for budget in (1, 0):  # 1 double: exactly the levels asked for
        print(f"[gpu] n={n} {pattern} mode={mode} budget={budget}", flush=True)
        caps_amd.set_available_memory(budget)
        C = torch.full_like(A, float("nan"))
        caps_amd.reset_counters()
        caps_amd.multiply_device(A, B, C, d, pattern, mode=mode, cutoff=cutoff)
        torch.cuda.synchronize()
        c = caps_amd.counters()
        want = "".join({"b": "BFS,", "d": "DFS,", "h": "HYB,"}[p] for p in pattern[:r - cutoff])
        assert c["pattern"] == want
        out.append((C, c["additions"], c["multiplications"], c["leaf_products"]))
        peak.append(c["peak_workspace_mb"])
    caps_amd.set_available_memory(0)
    assert torch.equal(out[0][0], out[1][0]) and out[0][1:] == out[1][1:]
    assert peak[1] > peak[0]  # the second did run batched
    N = torch.full_like(A, float("nan"))
    caps_amd.multiply_device_noalloc(A, B, N, d, pattern, mode=mode, cutoff=cutoff)
    torch.cuda.synchronize()
    assert torch.equal(N, out[0][0]) and caps_amd.counters()["pattern"] == want
    caps_amd.release()


@pytest.mark.parametrize("mode", [caps_amd.MODE_FP64, caps_amd.MODE_CRT_INT8])
@pytest.mark.parametrize("n,r,bs,pattern", [(1536, 2, 3, "dd"), (2048, 3, 1, "ddd")])
def test_levels_above_the_operands_size(n, r, bs, pattern, mode):
    """More workspace than the operands' size, little for the device."""
    test_small_recursive_levels(n, r, bs, pattern, 0, mode)
