"""One to three batched FP64 levels in single passes: the bits of the level-by-level
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
    _same_bits(m, pattern, bs, offset)


@pytest.mark.parametrize("m,pattern,bs,offset", [
    (1, "bb", 1, 1), (7, "bb", 1, 0), (49, "bb", 7, 1), (127, "bb", 1, 1), (128, "bb", 1, 0),
    (130, "bb", 5, 0), (257, "bb", 1, 0), (258, "bb", 3, 1), (35, "dbb", 5, 0)])
def test_two_levels_give_them_too(m, pattern, bs, offset):
    """Also at odd sizes and 8-byte alignment, plain and blocked leaves."""
    _same_bits(m, pattern, bs, offset)


@pytest.mark.parametrize("m,pattern,bs,offset", [
    (1, "b", 1, 0), (9, "b", 1, 1), (49, "b", 7, 0), (300, "b", 4, 1), (513, "b", 1, 0)])
def test_one_level_gives_them(m, pattern, bs, offset):
    _same_bits(m, pattern, bs, offset)


@pytest.mark.parametrize("m,pattern,bs", [
    (6, "bbbb", 3), (10, "bbbbb", 2), (260, "bbb", 4), (64, "bbb", 32), (20, "ddbb", 4)])
def test_blocked_leaves_below_further_levels(m, pattern, bs):
    """Leaves made column-major by the fused pass, further levels below it."""
    _same_bits(m, pattern, bs, 0)
    if len(pattern) < 4:
        _same_bits(m, pattern, bs, 0, caps_amd.MODE_OZAKI_INT8)


def _same_bits(m, pattern, bs, offset, mode=caps_amd.MODE_FP64):
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
        caps_amd.multiply_device(a, b, c, d, pattern, mode=mode, flags=flags)
        torch.cuda.synchronize()
        out.append(c)
    assert not torch.isnan(out[0]).any()
    assert torch.equal(out[0], out[1])
