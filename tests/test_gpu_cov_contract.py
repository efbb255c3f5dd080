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


@pytest.mark.parametrize("nspec", [1, 8])
def test_rows_and_contraction_meet(engine, nspec):
    """either side of the rule that picks the kernels: the same separations inside a plan that takes the
    contraction and, padded with further ones, a plan of so many that it takes the row transforms"""
    import torch
    from coffe_amd.covariance import CovPlan
    specs = batch_spectra(nspec, seed=4, lengths=(300,))
    k0 = specs[0][0]
    few = np.linspace(20.0, 150.0, 24) / H
    many = np.concatenate([few, np.linspace(20.3, 149.0, 900) / H])
    k = torch.tensor(np.concatenate([s[0] for s in specs]), device="cuda")
    p = torch.tensor(np.concatenate([s[1] for s in specs]), device="cuda")
    vals = []
    for sep in (few, many):
        plan = CovPlan(engine, 256, k0[0], k0[-1], LS, sep)
        out = plan.integrals(k, p, [300] * nspec)
        G = torch.zeros_like(out)
        G[..., :24, :24] = 1.0
        vals.append((out[..., :24, :24].cpu().numpy(), plan.integrals_vjp(k, p, [300] * nspec, G).cpu().numpy()))
        plan.close()
    (a, ga), (b, gb) = vals
    assert np.max(np.abs(a - b)) <= 1e-12 * np.max(np.abs(a))
    assert np.max(np.abs(ga - gb)) <= 1e-11 * np.max(np.abs(ga))
