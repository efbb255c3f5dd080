"""The two interval lists and the two spline lookups of the adaptive integrals
(quad_kernels.hip): integrals that outgrow the 64 intervals of the register list, spectra on
both sides of the LDS spline's 3000 samples, samples crowded into few index buckets, and more
integrals than one launch's wavefronts; against the oracle's QAG (the same bisections)."""
import numpy as np
import pytest

import oracle as O
from tests.synth import spectrum

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,spacing", [(60, "log"), (2999, "log"), (3000, "log"), (3001, "log"), (900, "linear"),
                                       (800, "clustered")])
def test_divergent_spline_lookup(engine, n, spacing):
    from coffe_amd.engine import divergent_tables
    k, _ = spectrum(n)
    if spacing == "linear":
        k = np.linspace(k[0], k[-1], n)
    elif spacing == "clustered":   # half of the samples inside one 64th of an octave
        k = np.sort(np.concatenate([k[:n // 2 * 2:2], 0.02 * (1 + 0.01 * np.linspace(0, 1, n - n // 2))]))
    pk = 2e4 * k / (1 + (k / 0.02) ** 2) ** 1.4
    sep = np.array([0.5, 7.0, 60.0, 400.0, 3000.0])
    chi = np.array([0.0, 12.0, 350.0, 2400.0])
    print(f"divergent n={n} {spacing}", flush=True)
    _, i40, r0, ren, status, nint = divergent_tables(k, pk, sep=sep, chi=chi, return_status=True)
    oi, orr, oren = O.divergent_tables(k, pk, sep, chi)
    # rounding of about 40 intervals of 61 values, against the largest value
    assert np.max(np.abs(i40 - oi)) <= 1e-12 * np.max(np.abs(oi))
    assert np.max(np.abs(ren - oren)) <= 1e-12 * np.max(np.abs(oren))
    assert np.max(np.abs(r0 / orr - 1)) <= 1e-10
    assert np.array_equal(ren, ren.T)


def test_long_interval_lists(engine):
    """the r = 0 renormalisation at tiny separations (1 - j0^2 near rounding): several hundred
    intervals, next to integrals of about twenty in the same launch"""
    from coffe_amd.engine import divergent_tables
    k, pk = spectrum(700)
    sep = np.array([1e-6, 5e-6, 1e-5, 0.5, 7.0, 60.0])
    chi = np.linspace(0.0, 2000.0, 50)
    _, i40, r0, ren, status, nint = divergent_tables(k, pk, sep=sep, chi=chi, return_status=True)
    ns = len(sep)
    assert nint[ns:2 * ns].max() > 64 and nint[2 * ns:].max() <= 64
    assert set(status.tolist()) <= {0, 1, 2}
    oi, orr, oren = O.divergent_tables(k, pk, sep, chi)
    assert np.max(np.abs(ren - oren)) <= 1e-12 * np.max(np.abs(oren))
    assert np.max(np.abs(i40[3:] / oi[3:] - 1)) <= 1e-11
    # below 1e-5 Mpc the integrand is rounding noise (1e-16 of 1 against x^2 / 3)
    assert np.max(np.abs(r0[3:] / orr[3:] - 1)) <= 1e-8


@pytest.mark.parametrize("nspec", [1, 7])
def test_small_r_few_and_many(engine, nspec):
    """one wavefront a workgroup (43 x 8 integrals) and eight (7 spectra), every order of the tables"""
    import torch
    from coffe_amd.engine import Batch
    tabs = [(0, 0), (0, 2), (0, 4), (1, 1), (1, 3), (2, 0), (2, 2), (3, 1)]
    ns = [300 + 500 * i for i in range(nspec)]
    specs = [spectrum(n) for n in ns]
    b = Batch(engine, ns, [512] * nspec, [s[0][0] for s in specs], [s[0][-1] for s in specs], tabs,
              np.array([20.0, 50.0]), 1, 1)
    got = b.small_r(torch.tensor(np.concatenate([s[0] for s in specs]), device="cuda"),
                    torch.tensor(np.concatenate([s[1] for s in specs]), device="cuda")).cpu().numpy()
    b.close()
    for s in {0, nspec - 1}:
        for t, (n, l) in enumerate(tabs):
            _, oy = O.integral_table(n, l, *specs[s], 512, small_r=True)
            assert np.all(np.abs(got[s, t] - oy[:43]) <= 1e-10 * np.abs(oy[:43]) + 1e-12 * np.max(np.abs(oy[:43]))), (n, l)


def test_small_r_shared_spline(engine):
    """eight wavefronts share one LDS spline: a batch whose spectra all fit (3000 samples, one short
    of that, a few dozen, the smallest), two tables and all eight; the longest sets the
    launch's LDS, the others fill a part of it"""
    import torch
    from coffe_amd.engine import Batch
    tabs = [(0, 0), (0, 2), (0, 4), (1, 1), (1, 3), (2, 0), (2, 2), (3, 1)]
    for ns, use in (([3000, 30, 600, 2999, 64, 5, 1200], tabs), ([40, 3000], tabs[3:5])):
        print("small r, shared spline", ns, flush=True)
        # the few samples over a narrow range: the integrands stay resolved
        specs = [spectrum(n, kmin=1e-5 if n > 50 else 0.02) for n in ns]
        b = Batch(engine, ns, [512] * len(ns), [s[0][0] for s in specs], [s[0][-1] for s in specs], use,
                  np.array([20.0, 50.0]), 1, 1)
        got = b.small_r(torch.tensor(np.concatenate([s[0] for s in specs]), device="cuda"),
                        torch.tensor(np.concatenate([s[1] for s in specs]), device="cuda")).cpu().numpy()
        b.close()
        for s in range(len(ns)):
            for t, (n, l) in enumerate(use):
                _, oy = O.integral_table(n, l, *specs[s], 512, small_r=True)
                assert np.all(np.abs(got[s, t] - oy[:43]) <= 1e-10 * np.abs(oy[:43]) + 1e-12 * np.max(np.abs(oy[:43]))), \
                    (ns[s], n, l)


def test_divergent_arguments_at_the_edges(engine):
    """chi so small that the product of two arguments underflows, next to 0 (j_0 is 1 at both); device
    arrays, whose signs are not checked: j_0 is even, so the integrals of -r are those of r (the
    factor r^4 is left out for r <= 0)"""
    import ctypes
    import torch
    from coffe_amd.engine import divergent_tables
    from coffe_amd._lib import check
    k, pk = spectrum(400)
    chi = np.array([0.0, 1e-300, 1e-170, 25.0, 900.0])
    _, _, _, ren = divergent_tables(k, pk, sep=np.array([5.0]), chi=chi)
    assert np.isfinite(ren).all()
    for i in (1, 2):
        assert np.array_equal(ren[i, 3:], ren[0, 3:]) and np.all(np.abs(ren[i, :3] / ren[0, 0] - 1) <= 1e-13)
    dev = dict(device="cuda", dtype=torch.float64)
    sep = np.array([7.0, -7.0, 60.0, -60.0])
    kt, pt, st = torch.tensor(k, **dev), torch.tensor(pk, **dev), torch.tensor(sep, **dev)
    i40, r0 = torch.zeros(4, **dev), torch.zeros(4, **dev)
    status = torch.zeros(8, dtype=torch.int32, device="cuda")
    check(engine.L.coffe_divergent_tables_device(engine.h, kt.data_ptr(), pt.data_ptr(), len(k), float(k[0]), float(k[-1]),
                                                 st.data_ptr(), 4, None, 0, i40.data_ptr(), r0.data_ptr(), None,
                                                 status.data_ptr(), None, ctypes.c_void_p(0)), "divergent")
    torch.cuda.synchronize()
    for v in (i40.cpu().numpy(), r0.cpu().numpy()):
        assert np.all(np.abs(v[1::2] * sep[::2] ** 4 / v[::2] - 1) <= 1e-13), v
