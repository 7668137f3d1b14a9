"""caps_multiply_device_noalloc with tables that do not fit beside the padded
workspace: copied in parts, the bits of caps_multiply_device."""
import pytest

import caps_amd

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,r,pattern,moduli", [(2176, 6, "ddddbb", 14), (2176, 7, "dddddbb", 8)])
def test_tables_in_parts(n, r, pattern, moduli):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    A, B = torch.rand((2, n * n), generator=g, device="cuda", dtype=torch.float64) * 2 - 1
    d = caps_amd.MatDescriptor.one_device(n, r, 1)
    out = []
    for entry in (caps_amd.multiply_device, caps_amd.multiply_device_noalloc):
        C = torch.full_like(A, float("nan"))
        for rep in range(2):  # the second call finds the plan and its parts
            print(f"[gpu] n={n} {pattern} {entry.__name__} {rep}", flush=True)
            C.fill_(float("nan"))
            entry(A, B, C, d, pattern, mode=caps_amd.MODE_CRT_INT8, moduli=moduli)
            torch.cuda.synchronize()
        out.append(C)
    assert not torch.isnan(out[0]).any() and torch.equal(out[0], out[1])
    caps_amd.release()
