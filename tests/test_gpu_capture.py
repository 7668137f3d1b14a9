"""Calls recorded into a caller's graph: every replay gives the eager result on new
operands, also after more other plans than the library keeps."""
import pytest

import caps_amd

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _setup():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    caps_amd.load()
    yield
    caps_amd.set_available_memory(0)
    caps_amd.release()


@pytest.mark.parametrize("entry", [caps_amd.multiply_device, caps_amd.multiply_device_noalloc])
@pytest.mark.parametrize("n,r,pattern,mode,budget", [
    (512, 2, "bb", caps_amd.MODE_FP64, 0), (640, 2, "bb", caps_amd.MODE_CRT_INT8, 0),
    (512, 2, "dd", caps_amd.MODE_CRT_INT8, 1)])  # as asked for: more than 16 launches
def test_replays_after_other_plans(n, r, pattern, mode, budget, entry):
    caps_amd.set_available_memory(budget)
    s = torch.cuda.Stream()
    A, B, C, want = torch.empty((4, n * n), device="cuda", dtype=torch.float64)
    d = caps_amd.MatDescriptor.one_device(n, r, 1)
    # plans of the same shape on other buffers
    others = torch.rand((30, 3, n * n), device="cuda", dtype=torch.float64)
    A.uniform_(-1, 1)
    B.uniform_(-1, 1)
    torch.cuda.synchronize()
    print(f"[gpu] capture n={n} {pattern} mode={mode} {entry.__name__}", flush=True)
    with torch.cuda.stream(s):
        entry(A, B, C, d, pattern, mode=mode)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        entry(A, B, C, d, pattern, mode=mode)
    for rep in range(4):
        A.uniform_(-1, 1)
        caps_amd.multiply_device(A, B, want, d, pattern, mode=mode)
        for o in others:
            entry(o[0], o[1], o[2], d, pattern, mode=mode)
        torch.cuda.synchronize()
        C.fill_(float("nan"))
        print(f"[gpu] replay {rep}", flush=True)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(C, want), rep
