"""Several tables of one spectrum in one call (coffe_integral_tables) against the tables one at a
time: lengths on the LDS kernels and on the general transform, windows inside the samples,
subsets and more than two biases; spline chunks of few and of many intervals."""
import numpy as np
import pytest

from tests.synth import spectrum

pytestmark = pytest.mark.gpu
TABLES = [(0, 0), (0, 2), (0, 4), (1, 1), (1, 3), (2, 0), (2, 2), (3, 1)]


@pytest.mark.parametrize("n,N,tables", [
    (600, 10000, TABLES), (40, 1024, TABLES), (5000, 1000, TABLES[:3]), (600, 16384, [(1, 3)]),
    (300, 1792, TABLES[:2]), (300, 40000, TABLES[2:4]), (300, 512, [(-1, 0), (0, 2), (4, 2), (0, 1)])])
def test_tables_at_once(engine, n, N, tables):
    from coffe_amd.engine import integral_table, integral_tables
    k, p = spectrum(n)
    for lo, hi in ((k[0], k[-1]), (k[2] * 1.01, k[-3] * 0.99)):
        print(f"integral_tables n={n} N={N} {tables}", flush=True)
        got = integral_tables(tables, k, p, N, lo, hi)
        assert list(got) == tables
        for t in tables:
            x, y = integral_table(*t, k, p, N, lo, hi)
            assert np.array_equal(got[t][0], x)
            # the same transforms; r^(n - l) multiplies in another order
            assert np.all(np.abs(got[t][1] - y) <= 1e-14 * np.abs(y) + 1e-16 * np.max(np.abs(y))), t


def test_refused_as_one_at_a_time(engine):
    from coffe_amd import EngineError
    from coffe_amd.engine import integral_table, integral_tables
    k, p = spectrum(300)
    bad = p.copy()
    bad[7] = np.nan
    for args in (((0, 0), k, p, 1001), ((0, 5), k, p, 1024), ((0, 0), k, bad, 1024), ((0, 0), k, p, 1024, k[0] / 2),
                 ((0, 0), k, p, 1024, k[5], k[5])):
        codes = []
        for call in (lambda t, *a: integral_table(*t, *a), lambda t, *a: integral_tables([t], *a)):
            with pytest.raises(EngineError) as err:
                call(*args)
            codes.append(err.value.code)
        assert codes[0] == codes[1], args


def test_no_grid_of_all_tables_where_they_go_one_by_one(engine):
    """at a length outside the LDS kernels the tables go one at a time, with their own grids: the joint call
    adds nothing to the device memory that those calls have taken"""
    import torch
    from coffe_amd.engine import integral_table, integral_tables
    k, p = spectrum(300)
    tables, N = TABLES[:3], 300000
    want = [integral_table(*t, k, p, N)[1] for t in tables]
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    got = integral_tables(tables, k, p, N)
    assert free - torch.cuda.mem_get_info()[0] < 1 << 20
    for t, w in zip(tables, want):
        assert np.array_equal(got[t][1], w)
