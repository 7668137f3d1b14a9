"""Three batched FP64 levels in single passes: the bits of the level-by-level
run (FLAG_NO_FUSION, the same expression trees) at odd and even leaf sizes, with
one position and with partly filled blocks, on both sides of the order from
which a thread takes all of a side, nested and below other levels, at operands
that are only 8-byte aligned."""
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


@pytest.mark.parametrize("m,pattern,bs,offset", [
    (1, "bbb", 1, 0), (3, "bbb", 3, 1), (16, "bbb", 1, 0), (49, "bbb", 7, 0), (90, "bbb", 1, 1),
    (255, "bbb", 1, 0), (256, "bbb", 1, 0), (257, "bbb", 1, 1), (5, "bbbb", 1, 0),
    (8, "bbbbb", 1, 1), (33, "dbbb", 1, 0), (10, "bbbd", 1, 0), (12, "bdbbb", 4, 1)])
def test_bits_of_the_level_by_level_run(m, pattern, bs, offset):
    r = len(pattern)
    n = m << r
    print(f"[gpu] m={m} {pattern} bs={bs} offset={offset}", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(m)
    a, b = (torch.rand(n * n + offset, generator=g, device="cuda", dtype=torch.float64)[offset:] - 0.5
            for _ in range(2))
    # a view of the generator's values keeps the offset
    a, b = (torch.cat([x.new_zeros(offset), x])[offset:] for x in (a, b))
    d = caps_amd.MatDescriptor.one_device(n, r, bs)
    out = []
    for flags in (0, caps_amd.FLAG_NO_FUSION):
        c = torch.full((n * n + offset,), float("nan"), device="cuda", dtype=torch.float64)[offset:]
        caps_amd.multiply_device(a, b, c, d, pattern, flags=flags)
        torch.cuda.synchronize()
        out.append(c)
    assert not torch.isnan(out[0]).any()
    assert torch.equal(out[0], out[1])
