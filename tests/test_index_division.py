"""The divisions of indices that the kernels replace by products: a frequency index by the box size (the rounded
reciprocal and one Newton step, in fused multiply-adds, rounds like the division for every index and size it is used
for) and an element index by a row length (a 32-bit multiplier and a shift)."""
import numpy as np
import pytest


@pytest.mark.parametrize("sizes", [(4096, 4097, 10007, 65535, 1 << 20), ((1 << 21) - 1, (1 << 22) - 3, (1 << 22) - 1)])
def test_newton_step_rounds_like_the_division_for_long_axes(sizes):
    """Axes of slices with fewer than 2^21 pixels: up to 2^22. The sum before the last rounding needs up to 72 bits and is
    formed in 64 here, which moves it by far less than its distance from a midpoint."""
    for n in sizes:
        i = np.arange(0, n + 1, dtype=np.float32)
        inv = np.float32(1) / np.float32(n)
        q = i * inv
        r = i.astype(np.longdouble) - q.astype(np.longdouble) * n
        assert (r.astype(np.float32) == r).all()
        got = (q.astype(np.longdouble) + r * np.longdouble(inv)).astype(np.float32)
        assert (got == i / np.float32(n)).all()


@pytest.mark.parametrize("sizes", [range(1, 1025), (1536, 2047, 2048, 3000, 4095)])
def test_newton_step_rounds_like_the_division(sizes):
    for n in sizes:
        i = np.arange(0, n + 1, dtype=np.float32)
        inv = np.float32(1) / np.float32(n)
        q = i * inv
        # A fused multiply-add of float32 values: exact in float64 (products of 24-bit values), then rounded once. The
        # last one rounds twice, which differs from once only where float64 falls on a float32 midpoint; none does.
        r = i.astype(np.float64) - q.astype(np.float64) * n
        assert (r.astype(np.float32) == r).all()
        got = (q.astype(np.float64) + r * np.float64(inv)).astype(np.float32)
        assert (got == i / np.float32(n)).all()


def test_element_index_quotient_is_exact():
    sizes = list(range(1, 2050)) + [4097, 65535, 65536, 65537, 2**30 - 1, 2**30, 2**30 + 1, 2**31 - 1]
    rng = np.random.default_rng(0)
    for d in sizes:
        shift = 31 + (d - 1).bit_length()
        mul = -(-(1 << shift) // d)
        assert mul < 1 << 32
        # The error grows with the index, so the last multiples below 2^31 and the index before each decide.
        last = (2**31 - 1) // d
        multiples = np.concatenate([np.arange(max(0, last - 64), last + 1), rng.integers(0, last + 1, 64)]) * d
        t = np.concatenate([multiples, multiples - 1, [2**31 - 1]])
        t = t[t >= 0].astype(np.uint64)
        assert ((t * np.uint64(mul)) >> np.uint64(shift) == t // np.uint64(d)).all(), d
