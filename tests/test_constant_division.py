"""Division by constants: the quotient of the division bit for bit."""
import numpy as np
import pytest

import parpy_amd as parpy

HIP = parpy.CompileBackend.Hip


def quotients(x, a, b, c, d, n):
    parpy.label('N')
    for i in range(n):
        a[i] = x[i] / 3.0
        b[i] = x[i] / 10.0
        c[i] = x[i] / -49.0
        d[i] = x[i] / 41.0


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=lambda d: np.dtype(d).name)
def test_division_by_a_constant_is_exact(dtype):
    """Quotients of all sizes in the normal range, zeros, infinities and NaN; below the normal range within one unit."""
    rng = np.random.default_rng(11)
    n = 1 << 20
    info = np.finfo(dtype)
    x = (rng.standard_normal(n) * np.exp2(rng.integers(info.minexp - 20, info.maxexp - 2, n).astype(np.float64))).astype(dtype)
    x[:8] = [0.0, -0.0, np.inf, -np.inf, np.nan, info.max, -info.max, info.smallest_subnormal]
    out = [np.zeros(n, dtype=dtype) for _ in range(4)]
    o = parpy.par({'N': parpy.threads(n)})
    o.backend = HIP
    parpy.jit(quotients)(x, *out, n, opts=o)
    with np.errstate(all="ignore"):
        for c, got in zip((3.0, 10.0, -49.0, 41.0), out):
            want = x / dtype(c)
            normal = ~(np.abs(want) < info.tiny) | (want == 0)
            assert np.array_equal(want[normal], got[normal], equal_nan=True), c
            number = ~np.isnan(want)
            assert np.array_equal(np.signbit(want[number]), np.signbit(got[number]))
            assert np.abs(want[~normal] - got[~normal]).max() <= info.smallest_subnormal, c
