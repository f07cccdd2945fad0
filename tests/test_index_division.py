"""The division of a frequency index by the box size in the rasterisation: a product with the rounded reciprocal and one
Newton step, in fused multiply-adds, rounds like the division for every index and size it is used for."""
import numpy as np
import pytest


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
