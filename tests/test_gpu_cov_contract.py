"""The contraction kernels of the covariance integrals (k_cov_many / k_cov_few and their
transposes) at the edges of their tiles: 16 separations, 16 diagonals (two per
spectrum), 16 k nodes, 64 separations per wave of the adjoint, lengths outside the LDS
transforms; sorted and unsorted separations.

- integrals of the first and the last spectrum against the oracle's 2D transform, 1e-10 of the
  block's largest value (as the other covariance tests);
- the batch against one spectrum at a time (the other kernel, another order of the sums over N
  terms): 1e-12 of the largest value, N eps with room for the cancellation in the sums;
- the adjoint: Euler's identity sum gpk P = <G1, I1> + 2 <G2, I2> (the integrals of P and P^2 are
  homogeneous of degree 1 and 2 in the samples), 1e-11 of sum |gpk P|, and the batch against
  single spectra, 1e-11 of the largest gradient (Akima's weights amplify the sums' rounding)."""
import numpy as np
import pytest

import oracle as O
from tests.synth import batch_spectra

pytestmark = pytest.mark.gpu

H = 0.67
LS = [0, 2]


@pytest.mark.parametrize("nspec,N,R,order", [
    (1, 256, 1, "up"), (1, 250, 17, "mixed"), (4, 128, 65, "up"), (2, 126, 16, "down"),
    (5, 250, 15, "up"), (8, 256, 16, "mixed"), (9, 200, 33, "up"), (20, 128, 31, "down"), (64, 256, 20, "up")])
def test_contraction_vs_oracle_and_single(engine, nspec, N, R, order):
    import torch
    from coffe_amd.covariance import CovPlan
    specs = batch_spectra(nspec, seed=nspec + R, lengths=(300,))
    k0 = specs[0][0]
    sep = np.linspace(12.0, 180.0, R) / H if R > 1 else np.array([77.0])
    sep = {"up": sep, "down": sep[::-1].copy(), "mixed": np.random.default_rng(R).permutation(sep)}[order]
    plan = CovPlan(engine, N, k0[0], k0[-1], LS, sep)
    plan.set_path("contract")
    print(f"contraction nspec={nspec} N={N} R={R} {order}", flush=True)
    k = torch.tensor(np.concatenate([s[0] for s in specs]), device="cuda")
    p = torch.tensor(np.concatenate([s[1] for s in specs]), device="cuda")
    n_in = [300] * nspec
    got = plan.integrals(k, p, n_in).cpu().numpy()
    for s in {0, nspec - 1}:
        for power in (1, 2):
            for q, (i, j) in enumerate(plan.pairs):
                ref = O.covariance_fftlog_integral(specs[s][0], specs[s][1], float(power), LS[i], LS[j], N, sep, k0[0],
                                                   k0[-1])
                ref = ref * (2 * LS[i] + 1) * (2 * LS[j] + 1) * (2.0 if power == 1 else 1.0) / np.pi ** 2
                assert np.max(np.abs(got[s, power - 1, q] - ref)) <= 1e-10 * np.max(np.abs(ref)), (s, power, q)
        one = plan.integrals(k[300 * s:300 * s + 300], p[300 * s:300 * s + 300], [300]).cpu().numpy()[0]
        assert np.max(np.abs(one - got[s])) <= 1e-12 * np.max(np.abs(one))
    assert plan.path == "contract"
    if N == 126:   # 2 3^2 7: no adjoint outside the LDS lengths
        plan.close()
        return
    G = torch.tensor(np.random.default_rng(3).standard_normal(got.shape), device="cuda")
    gpk = plan.integrals_vjp(k, p, n_in, G).cpu().numpy().reshape(nspec, -1)
    P = p.cpu().numpy().reshape(nspec, -1)
    w = (G.cpu().numpy() * got * np.array([1.0, 2.0])[None, :, None, None, None]).reshape(nspec, -1).sum(axis=1)
    assert np.all(np.abs((gpk * P).sum(axis=1) - w) <= 1e-11 * np.abs(gpk * P).sum(axis=1))
    for s in {0, nspec - 1}:
        one = plan.integrals_vjp(k[300 * s:300 * s + 300], p[300 * s:300 * s + 300], [300],
                                 G[s:s + 1].contiguous()).cpu().numpy()
        assert np.max(np.abs(one - gpk[s])) <= 1e-11 * np.max(np.abs(one))
    plan.close()


def _spectra(nspec, n=300, seed=4):
    import torch
    specs = batch_spectra(nspec, seed=seed, lengths=(n,))
    k = torch.tensor(np.concatenate([s[0] for s in specs]), device="cuda")
    p = torch.tensor(np.concatenate([s[1] for s in specs]), device="cuda")
    return specs[0][0], k, p, [n] * nspec


@pytest.mark.parametrize("nspec,N,R", [(1, 256, 924), (8, 256, 924), (3, 1000, 300), (2, 1792, 40), (9, 250, 70)])
def test_rows_and_contraction_meet(engine, nspec, N, R):
    """either side of the rule that picks the kernels: the same plan both ways, the sums over N terms in
    another order (as above); separations in no order, lengths with a factor 7 (no adjoint)"""
    import torch
    from coffe_amd.covariance import CovPlan
    k0, k, p, n_in = _spectra(nspec)
    sep = np.random.default_rng(R).permutation(np.linspace(20.0, 150.0, R) / H)
    plan = CovPlan(engine, N, k0[0], k0[-1], LS, sep)
    print(f"rows and contraction nspec={nspec} N={N} R={R}", flush=True)
    vals = []
    for path in ("rows", "contract"):
        plan.set_path(path)
        out = plan.integrals(k, p, n_in)
        assert plan.path == path
        g = None
        if N != 1792:
            G = torch.randn(out.shape, dtype=torch.float64, device="cuda", generator=torch.Generator("cuda").manual_seed(1))
            g = plan.integrals_vjp(k, p, n_in, G).cpu().numpy()
            assert plan.path == path
        vals.append((out.cpu().numpy(), g))
    plan.close()
    (a, ga), (b, gb) = vals
    assert np.max(np.abs(a - b)) <= 1e-12 * np.max(np.abs(a))
    if ga is not None:
        assert np.max(np.abs(ga - gb)) <= 1e-11 * np.max(np.abs(ga))


def test_the_rule_takes_both(engine):
    """without a choice: few separations are a contraction, many of one spectrum row transforms"""
    from coffe_amd.covariance import CovPlan
    k0, k, p, n_in = _spectra(1)
    for R, path in ((24, "contract"), (924, "rows")):
        plan = CovPlan(engine, 256, k0[0], k0[-1], LS, np.linspace(20.0, 150.0, R) / H)
        assert plan.path == "auto"
        plan.integrals(k, p, n_in)
        assert plan.path == path
        plan.close()


@pytest.mark.parametrize("nspec", [4, 8])
def test_workspace_is_bounded(engine, nspec):
    """470 separations of 4 spectra: 8 splits of 48 integrals are 680 MB, so k_cov_few takes the integrals in
    two launches; of 8 spectra, k_cov_many takes fewer splits.  Against the row transforms, and
    the device memory that a call adds (512 MB, the diagonals, and some slack for the pool)."""
    import torch
    from coffe_amd.covariance import CovPlan
    k0, k, p, n_in = _spectra(nspec)
    plan = CovPlan(engine, 256, k0[0], k0[-1], [0, 2, 4], np.linspace(20.0, 150.0, 470) / H)
    out = torch.zeros((nspec, 2, plan.npair, 470, 470), dtype=torch.float64, device="cuda")
    plan.set_path("contract")
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    got = plan.integrals(k, p, n_in, out=out).cpu().numpy()
    assert plan.path == "contract" and free - torch.cuda.mem_get_info()[0] <= 540 << 20
    plan.set_path("rows")
    ref = plan.integrals(k, p, n_in).cpu().numpy()
    plan.close()
    assert np.max(np.abs(got - ref)) <= 1e-12 * np.max(np.abs(ref))


def test_rows_where_memory_is_short(engine):
    """each allocation of a plan's tables and of a call's workspaces failing in turn: what the row
    transforms can do without it, they do (the same values as when chosen; their adjoint adds
    atomically, so to 1e-11 as above), and the rest is ENOMEM; a plan without tables makes them in the first call that has room"""
    import torch
    from coffe_amd import EngineError
    from coffe_amd.covariance import CovPlan
    L = engine.L
    k0, k, p, n_in = _spectra(1)
    sep = np.linspace(20.0, 150.0, 24) / H
    args = (engine, 256, k0[0], k0[-1], LS, sep)
    plan = CovPlan(*args)
    ref = {}
    for path in ("rows", "contract"):
        plan.set_path(path)
        out = plan.integrals(k, p, n_in)
        ref[path] = (out.cpu().numpy(), plan.integrals_vjp(k, p, n_in, torch.ones_like(out)).cpu().numpy())
    G = torch.ones_like(out)
    plan.close()
    went = []

    def same(a, b):
        assert np.max(np.abs(a.cpu().numpy() - b)) <= (1e-11 if b.ndim == 1 else 0.0) * np.max(np.abs(b))

    try:
        for call in (0, 1):
            for n in range(1, 20):
                plan = CovPlan(*args)
                if call:
                    plan.integrals(k, p, n_in)
                L.coffe_engine_inject_alloc_failure(n)
                try:
                    got = plan.integrals_vjp(k, p, n_in, G) if call else plan.integrals(k, p, n_in)
                except EngineError as err:
                    assert err.code == 2
                    went.append("enomem")
                    plan.close()
                    continue
                finally:
                    L.coffe_engine_inject_alloc_failure(0)
                went.append(plan.path)
                same(got, ref[plan.path][call])
                out = plan.integrals(k, p, n_in)   # and the plan goes on
                same(out, ref[plan.path][0])
                plan.close()
                if went[-1] == "contract":
                    break
        assert went.count("contract") == 2 and went.count("rows") >= 3, went
        # the tables themselves, when the plan is made: the first call makes them
        made = 0
        for n in range(1, 60):
            L.coffe_engine_inject_alloc_failure(n)
            try:
                plan = CovPlan(*args)
            except EngineError as err:
                assert err.code == 2
                continue
            finally:
                L.coffe_engine_inject_alloc_failure(0)
            made += 1
            got = plan.integrals(k, p, n_in)
            assert plan.path == "contract"
            same(got, ref["contract"][0])
            plan.close()
            # without room in that call either the plan keeps to the rows
            if made <= 3:
                L.coffe_engine_inject_alloc_failure(n)
                plan = CovPlan(*args)
                L.coffe_engine_inject_alloc_failure(4)   # the spectra's three, then the tables'
                got = plan.integrals(k, p, n_in)
                L.coffe_engine_inject_alloc_failure(0)
                assert plan.path == "rows"
                same(got, ref["rows"][0])
                plan.integrals(k, p, n_in)
                assert plan.path == "rows"
                plan.close()
            if made == 4:
                break
        assert made == 4
    finally:
        L.coffe_engine_inject_alloc_failure(0)
