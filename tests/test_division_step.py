"""Divisions of the KIVI quantisation ladder (quant_pack.py's bf16 ladder,
S:2003-2009) and of rabitq4.hip's encode.  The kernels need bf16(x / b) of two
bf16 values and take it as bf16(x * (1 / b)) (csrc/zkv_common.hpp, kivi_code
and kivi_scale).

While quotient and reciprocal are normal, the rounding of every step depends
only on the operands' significands (scaling x or b by a power of two scales
every intermediate by the same power), so every pair of bf16 significands
covers every pair of normal bf16 operands; x / 15 is checked for every bf16 x.
"""
import numpy as np


def _bf16_from_bits(bits: np.ndarray) -> np.ndarray:
    return (bits.astype(np.uint32) << 16).view(np.float32)


def _bf16_rne(x: np.ndarray) -> np.ndarray:
    u = x.astype(np.float32).view(np.uint32).astype(np.uint64)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint32)


def _significand_pairs(ex: int, ed: int):
    sig = 1.0 + np.arange(128, dtype=np.float64) / 128.0
    xs, ds = np.meshgrid(sig, sig, indexing="ij")
    return np.ldexp(xs, ex).astype(np.float32), np.ldexp(ds, ed).astype(np.float32)


def _by_product(x: np.ndarray, r: np.ndarray) -> np.ndarray:
    with np.errstate(over="ignore"):
        return _bf16_rne((x * r).astype(np.float32))


def _by_division(x: np.ndarray, d: np.ndarray) -> np.ndarray:
    with np.errstate(over="ignore"):
        return _bf16_rne(x / d)


def test_every_bf16_over_15_by_reciprocal_product():
    """Signs, zeros, subnormals and infinities included (NaN stays NaN)."""
    x = _bf16_from_bits(np.arange(0x10000, dtype=np.uint32))
    with np.errstate(invalid="ignore"):
        got, want = _by_product(x, np.float32(1.0 / 15.0)), _by_division(x, np.float32(15.0))
    num = ~np.isnan(x)
    assert np.array_equal(got[num], want[num])
    assert np.isnan(_bf16_from_bits(got[~num])).all()


def test_bf16_quotient_by_reciprocal_product():
    """Every pair of significands, with quotients from overflow down through
    bf16's subnormal range, and with the reciprocal off by one unit in the
    last place (the hardware's) where the quotient is normal."""
    for ex, ed in [(0, 0), (127, 0), (127, -1), (127, -26), (-60, 67), (100, 127), (-126, 0)] + \
            [(-60, e) for e in range(63, 80)]:
        x, d = _significand_pairs(ex, ed)
        ref = _by_division(x, d)
        r = (np.float32(1.0) / d).astype(np.float32)
        assert np.array_equal(_by_product(x, r), ref), (ex, ed)
        if -100 < ex - ed < 120:
            for to in (np.float32(0), np.float32(np.inf)):
                assert np.array_equal(_by_product(x, np.nextafter(r, to)), ref), (ex, ed, to)


def test_a_worse_reciprocal_is_noticed():
    """Planted: a reciprocal off by 2^-16 of itself (128 to 256 units in the
    last place) crosses the midpoint of some pair, upwards and downwards, so
    the exact comparison above can fail; so does one rounded to bf16."""
    x, d = _significand_pairs(0, 0)
    ref = _by_division(x, d)
    r = (np.float32(1.0) / d).astype(np.float32)
    for off in (2.0 ** -16, -2.0 ** -16):
        assert (_by_product(x, (r * np.float32(1.0 + off)).astype(np.float32)) != ref).any(), off
    assert (_by_product(x, _bf16_from_bits(_bf16_rne(r))) != ref).any()
