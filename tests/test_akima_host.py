"""coffe_akima_eval on the host: the coefficients of all intervals (a third as many queries as nodes, or
more) and of the queries' intervals only (fewer) give the same bits, and the oracle's values."""
import ctypes

import numpy as np
import pytest

import oracle as O


def _eval(x, y, q):
    from coffe_amd._lib import load_library
    dp = ctypes.POINTER(ctypes.c_double)
    out = np.empty(len(q))
    f = load_library().coffe_akima_eval
    f.argtypes = [ctypes.c_size_t, dp, dp, ctypes.c_size_t, dp, dp]
    assert f(len(x), x.ctypes.data_as(dp), y.ctypes.data_as(dp), len(q), q.ctypes.data_as(dp), out.ctypes.data_as(dp)) == 0
    return out


@pytest.mark.parametrize("n", [5, 6, 29, 400])
@pytest.mark.parametrize("shape", ["noise", "steps", "flat"])
def test_few_and_many_queries(n, shape):
    rng = np.random.default_rng(n)
    x = np.cumsum(rng.uniform(0.1, 2.0, n))
    y = {"noise": rng.standard_normal(n), "steps": np.floor(np.arange(n) / 3.0), "flat": np.full(n, 2.5)}[shape]
    q = np.concatenate([x, (x[1:] + x[:-1]) / 2, rng.uniform(x[0], x[-1], 50), [x[0] - 1, x[-1] + 1, np.nan]])
    many = _eval(x, y, q)
    one = np.array([_eval(x, y, q[i:i + 1])[0] for i in range(len(q))])
    assert np.array_equal(many, one, equal_nan=True)
    assert np.isnan(many[-3:]).all() and np.isfinite(many[:-3]).all()
    # a few operations on values of order one
    assert np.max(np.abs(many[:-3] - O.akima(x, y, q[:-3]))) <= 1e-13 * (1 + np.max(np.abs(y)))
