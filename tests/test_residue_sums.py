"""The leaf GEMMs' exact reductions modulo m (residue_of_sum and
residue_of_f32 in caps_amd/csrc/ozaki_dev.h), restated in numpy with the same
FP32 rounding and checked for every modulus over every value their float part
can see.  An FP32 fma of an FP32 product and addend is one rounding of a value
that float64 holds exactly."""
import numpy as np

from oracle import split

MAGIC = 12582912  # 1.5 * 2^23


def low_byte(x, m):
    """round(x / m) through the low bits of fma(x, 1/m, MAGIC), then x - k m as
    the low byte of a 24-bit multiply-add of those bits."""
    inv = np.float32(1.0) / np.float32(m)
    assert np.array_equal(x.astype(np.float32).astype(np.int64), x)  # exact in FP32
    t = (x.astype(np.float64) * np.float64(inv) + MAGIC).astype(np.float32)
    bits = t.view(np.int32).astype(np.int64) & 0xFFFFFF  # mad24 reads 24 bits, sign bit clear
    assert bits.max() < 1 << 23 and bits.min() >= 0
    return (bits * -m + x) & 0xFF


def want(x, m):
    return (np.mod(x + m // 2, m) - m // 2) & 0xFF


def consts(m):
    c16 = (1 << 16) % m
    bias = -(-(1 << 28) // m) * m
    return c16, bias


def test_every_folded_sum():
    # xb = x + bias < 2^29 + 256, so y <= 65535 + 8192 * 255 < 2^21.1
    for m in split.moduli(16):
        c16, bias = consts(m)
        assert bias % m == 0 and bias >= 1 << 28 and bias + (1 << 28) < 1 << 31
        top = 65535 + ((bias + (1 << 28)) >> 16) * c16
        y = np.arange(0, top + 1, dtype=np.int64)
        assert np.array_equal(low_byte(y, m), want(y, m)), m


def test_the_dot_product_folds_exactly():
    rng = np.random.default_rng(3)
    x = np.concatenate([rng.integers(-(1 << 28), (1 << 28) + 1, 1_000_000),
                        [-(1 << 28), (1 << 28), 0, -1, 1]])
    for m in split.moduli(16):
        c16, bias = consts(m)
        xb = x + bias
        assert xb.min() >= 0
        y = (xb & 0xFFFF) + (xb >> 16) * c16
        assert np.array_equal(np.mod(y - x, m), np.zeros_like(y)), m
        assert np.array_equal(low_byte(y, m), want(x, m)), m


def test_every_fp32_sum():
    # a folded sum (1.5 m) and 512 products of at most 2^14
    for m in split.moduli(16):
        top = (1 << 23) + (3 * m) // 2
        for lo in range(-top, top + 1, 1 << 21):
            x = np.arange(lo, min(lo + (1 << 21), top + 1), dtype=np.int64)
            assert np.array_equal(low_byte(x, m), want(x, m)), (m, lo)


def test_not_vacuous():
    """Well past the range the one-step quotient fails."""
    x = np.arange((1 << 27) - 4096, 1 << 27, 8, dtype=np.int64)
    assert not np.array_equal(low_byte(x, 199), want(x, 199))
