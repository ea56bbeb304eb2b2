"""FP32 quotients as the multigrid kernels form them, n / d = (float)(n * (1 / d))
with the reciprocal and the product in FP64, against FP32 division.

Two 24-bit significands' quotient is at least 2^-49 (relative) away from the
middle between two floats, and the reciprocal and the product are off by 2^-52 and
2^-53, so the results are equal; below the normal numbers the middles are
coarser and can be hit exactly, where either neighbour is half a step away.
"""
from __future__ import annotations

import numpy as np
import pytest


@pytest.mark.parametrize("ne,de", [(0, 0), (-100, 10), (-126, 0), (-149, 3), (100, 126), (0, 127), (-20, -126),
                                   (-30, -140), (-100, 49)])
@pytest.mark.parametrize("off", [-1, 0, 1])  # ulps of the reciprocal
def test_equals_division(ne, de, off):
    rng = np.random.default_rng(7)
    m = 200000
    n = (rng.uniform(1.0, 2.0, m) * 2.0 ** ne * rng.choice([-1.0, 1.0], m)).astype(np.float32)
    d = (rng.uniform(1.0, 2.0, m) * 2.0 ** de).astype(np.float32)
    n, d = n[d != 0], d[d != 0]
    with np.errstate(all="ignore"):
        y = 1.0 / d.astype(np.float64)
        y = y * (1.0 + off * 2.0 ** -52)
        got = (n.astype(np.float64) * y).astype(np.float32)
        want = n / d
        exact = n.astype(np.longdouble) / d.astype(np.longdouble)
    same = got == want
    step = np.longdouble(2.0 ** -149)
    tie = np.abs(np.abs(got - exact) - step / 2) <= step * 2.0 ** -40
    assert (same | (tie & (np.abs(want) < 2.0 ** -126))).all()
    assert same.mean() > 0.9
