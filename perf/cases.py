"""Performance cases of the multiply: what a program that uses this library has
it do, over the sizes, depths, layouts and leaf modes it is used at.

listed()            the cases, each a dict of plain values
draw(rng)           one more case of the same ranges
prepare(case, seed) operands of that seed, in the layout the call takes
run(state)          one pass through the public entry points
work(case)          bytes and operations a pass cannot do without
exact(case, seed)   the same outputs from plain FP64 torch / numpy

Case fields: "do" (multiply: device-resident operands; host: the drop-in call
on host arrays; batch: independent problems in one call; layout: column-major
to the CAPS layout and back), "n" the order, "nrec" the layout's quadrant
levels, "bs" its block size, "mode" the leaf arithmetic (fp64, auto: the
library chooses, crt: INT8 residues, bf16: the residues on BF16), "pattern"
(auto: the library chooses; reference: the one-process rule of the reference,
recursive at every level; else one char per level), "spread": entries are
u * 2^e, u uniform in [-1, 1), e a uniform integer in [-spread, spread].  A
batch has "count" problems with n up to "n" from the size generator "sizes".
"""
import math

import numpy as np
import torch

import caps_amd
from caps_amd import batch_plan

MODES = {"fp64": caps_amd.MODE_FP64, "auto": caps_amd.MODE_AUTO,
         "crt": caps_amd.MODE_CRT_INT8, "bf16": caps_amd.MODE_CRT_BF16}


def case(name, do, n, nrec, bs=1, mode="fp64", pattern="auto", spread=0, count=1, sizes=0):
    c = {"do": do, "n": n, "nrec": nrec, "bs": bs, "mode": mode, "pattern": pattern,
         "spread": spread, "count": count, "sizes": sizes}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the reference's fixture shape (leaves of 49 in blocks of 7): the
        # smallest call, all latency
        case("fp64 392 bdd bs7", "multiply", 392, 3, 7, "fp64", "bdd"),
        # a small multiply with every default: one of many in a larger program
        case("fp64 1024", "multiply", 1024, 2),
        # the drop-in call as the reference's callers make it: host arrays in,
        # host array out
        case("host 2048", "host", 2048, 2),
        # the reference's own one-process choice (recursive at every level) at
        # an ordinary size
        case("fp64 4096 reference", "multiply", 4096, 3, 1, "fp64", "reference"),
        # an order that is a multiple of nothing convenient: leaves of 625
        case("fp64 5000 ragged", "multiply", 5000, 3),
        # the benchmark's plain FP64 multiply
        case("fp64 8192 bb", "multiply", 8192, 2, 1, "fp64", "bb", 10),
        # the accurate mode the library chooses by itself, at a small size
        case("auto 1280", "multiply", 1280, 2, 1, "auto", "auto", 10),
        # residues on a ragged order: leaves of 750
        case("crt 3000 ragged", "multiply", 3000, 2, 1, "crt", "auto", 10),
        # the benchmark's headline multiply
        case("crt 8192 bb", "multiply", 8192, 2, 1, "crt", "bb", 10),
        # the BF16 form of the same arithmetic
        case("bf16 4096 bb", "multiply", 4096, 2, 1, "bf16", "bb", 10),
        # independent problems of uneven sizes in one call
        case("batch crt 32", "batch", 2048, 0, 1, "crt", "auto", 0, 32, 2024),
        # a column-major matrix into the layout and back, small blocks
        case("layout 8192 bs8", "layout", 8192, 2, 8),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _order(rng, lo, hi, nrec):
    """An order near a log-uniform target: 2^nrec leaves of a size that is a
    multiple of 1 (odd ones among them), 2, 16 or 64."""
    grain = rng.choice([1, 2, 16, 64])
    m = max(1, round(_log(rng, lo, hi) / (1 << nrec) / grain)) * grain
    return m << nrec


def _block(rng, n, nrec):
    """Mostly bs = 1 (column-major leaves), else a small divisor of the leaf."""
    m = n >> nrec
    divisors = [b for b in (2, 4, 5, 7, 8, 16, 32, 64) if m % b == 0]
    return rng.choice(divisors) if divisors and rng.random() < 0.25 else 1


def draw(rng):
    do = rng.choice(["multiply"] * 7 + ["host", "batch", "layout"])
    nrec = rng.choice([1, 2, 2, 3])
    if do == "layout":
        n = _order(rng, 512, 8192, nrec)
        return case(None, do, min(n, 8192), nrec, _block(rng, min(n, 8192), nrec))
    if do == "batch":
        return case(None, do, rng.choice([1024, 1536, 2048]), 0, 1, rng.choice(["fp64", "crt"]),
                    "auto", 0, rng.randint(8, 48), rng.randint(1, 10 ** 6))
    if do == "host":
        n = _order(rng, 400, 2400, nrec)
        return case(None, do, n, nrec, _block(rng, n, nrec))
    mode = rng.choice(["fp64"] * 4 + ["auto", "crt", "crt", "bf16"])
    # the residue modes on leaves of an odd size, and BF16, cost several times
    # an aligned multiply of that order: drawn up to half the largest
    hi = {"fp64": 8000, "bf16": 4200}.get(mode, 7600 if rng.random() < 0.5 else 4000)
    n = _order(rng, 300, hi, nrec)
    if mode != "fp64" and (n >> nrec) % 16 and n > 4200:
        n = ((n >> nrec) // 64 * 64) << nrec
    pattern = rng.choice(["auto", "auto", "reference", "given"])
    if pattern == "given":
        pattern = "".join(rng.choice("bd") for _ in range(nrec))
    bs = _block(rng, n, nrec)
    return case(None, do, n, nrec, bs, mode, pattern, rng.choice([0, 10]))


# ------------------------------------------------------------------ operands
def _problems(c):
    """(n, nrec, pattern) of every problem of the case."""
    if c["do"] != "batch":
        return [(c["n"], c["nrec"], c["pattern"])]
    sizes = batch_plan.uneven_sizes(c["count"], c["sizes"], 128, c["n"])
    plans = [batch_plan.default_plan(n, caps_amd.DEFAULT_MODULI) for n in sizes]
    return [(n, p.nrec, p.pattern) for n, p in zip(sizes, plans)]


def _entries(n, spread, g):
    u = torch.rand(n * n, generator=g, device="cuda", dtype=torch.float64) * 2 - 1
    if spread:
        e = torch.randint(-spread, spread + 1, (n * n,), generator=g, device="cuda",
                          dtype=torch.int32)
        u = torch.ldexp(u, e.to(torch.float64))
    return u


def _host_entries(n, seed):
    rng = np.random.default_rng(seed)
    return rng.uniform(-1.0, 1.0, (2, n * n))


def prepare(case, seed):
    s = {"do": case["do"], "mode": MODES[case["mode"]], "flags": 0}
    if case["do"] == "host":
        A, B = _host_entries(case["n"], seed)
        s.update(A=A, B=B, C=np.empty_like(A), pattern=None,
                 desc=caps_amd.MatDescriptor.one_device(case["n"], case["nrec"], case["bs"]))
        return s
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    probs = _problems(case)
    s["desc"] = [caps_amd.MatDescriptor.one_device(n, r, case["bs"]) for n, r, _ in probs]
    s["A"] = [_entries(n, case["spread"], g) for n, _, _ in probs]
    if case["do"] == "layout":
        s["caps"], s["back"] = torch.empty_like(s["A"][0]), torch.empty_like(s["A"][0])
        return s
    s["B"] = [_entries(n, case["spread"], g) for n, _, _ in probs]
    s["C"] = [torch.empty_like(a) for a in s["A"]]
    s["pattern"] = [None if p in ("auto", "reference") else p for _, _, p in probs]
    if case["pattern"] == "reference":
        s["flags"] = caps_amd.FLAG_REFERENCE_AUTO
    return s


def run(s):
    if s["do"] == "host":
        caps_amd.multiply(s["A"], s["B"], s["C"], s["desc"], s["pattern"], mode=s["mode"])
        return s["C"]
    if s["do"] == "layout":
        caps_amd.to_layout_device(s["A"][0], s["caps"], s["desc"][0])
        caps_amd.from_layout_device(s["caps"], s["back"], s["desc"][0])
        return [s["caps"], s["back"]]
    if s["do"] == "batch":
        caps_amd.multiply_batch_device(s["A"], s["B"], s["C"], s["desc"], s["pattern"],
                                       mode=s["mode"])
        return s["C"]
    caps_amd.multiply_device(s["A"][0], s["B"][0], s["C"][0], s["desc"][0], s["pattern"][0],
                             mode=s["mode"], flags=s["flags"])
    return s["C"][0]


# ------------------------------------------------------------------ the floor and the truth
def work(case):
    """Bytes: operands read and the result written once.  Operations: the
    additions and the leaf products of nrec Winograd levels; in the residue
    modes the leaf products modulo 14 moduli."""
    if case["do"] == "layout":
        return {"bytes": 32 * case["n"] ** 2, "flops": 0}
    nbytes = flops = 0
    for n, r, _ in _problems(case):
        nbytes += 24 * n * n
        leaf = 2 * 7 ** r * (n >> r) ** 3
        if case["mode"] == "fp64":
            flops += leaf + sum(7 ** k * 15 * (n >> (k + 1)) ** 2 for k in range(r))
        else:
            flops += caps_amd.DEFAULT_MODULI * leaf
    return {"bytes": nbytes, "flops": flops}


def _dims(n, nrec, bs):
    """Shape of a CAPS-layout vector with one axis per quadrant bit (column
    then row, outermost level first), then block column, block row, column and
    row in the block; and the axes in (column, row) order."""
    nb = (n >> nrec) // bs
    shape = [2, 2] * nrec + [nb, nb, bs, bs]
    cols = [2 * k for k in range(nrec)] + [2 * nrec, 2 * nrec + 2]
    rows = [2 * k + 1 for k in range(nrec)] + [2 * nrec + 1, 2 * nrec + 3]
    return shape, cols + rows


def _to_columns(v, n, nrec, bs):
    """CAPS-layout vector -> n x n tensor indexed [column, row]."""
    shape, axes = _dims(n, nrec, bs)
    return v.reshape(shape).permute(axes).reshape(n, n)


def _to_caps(m, n, nrec, bs):
    """n x n tensor indexed [column, row] -> CAPS-layout vector."""
    shape, axes = _dims(n, nrec, bs)
    inverse = [axes.index(k) for k in range(len(axes))]
    return m.reshape([shape[k] for k in axes]).permute(inverse).reshape(-1).contiguous()


def exact(case, seed):
    bs = case["bs"]
    if case["do"] == "host":
        A, B = (torch.from_numpy(x) for x in _host_entries(case["n"], seed))
        n, r = case["n"], case["nrec"]
        C = _to_columns(B, n, r, bs) @ _to_columns(A, n, r, bs)  # (A B)^T by columns
        return _to_caps(C, n, r, bs).numpy()
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    probs = _problems(case)
    A = [_entries(n, case["spread"], g) for n, _, _ in probs]
    if case["do"] == "layout":
        n, r, _ = probs[0]
        return [_to_caps(A[0].reshape(n, n), n, r, bs), A[0]]
    B = [_entries(n, case["spread"], g) for n, _, _ in probs]
    C = [_to_caps(_to_columns(b, n, r, bs) @ _to_columns(a, n, r, bs), n, r, bs)
         for a, b, (n, r, _) in zip(A, B, probs)]
    return C if case["do"] == "batch" else C[0]
