"""The double integral's two variants (k_integrated_double): tables on shared nodes are
fetched a line at a time by the whole wavefront; tables on nodes of their own, I_0^4 or
renormalisation grids too large for LDS (512 nodes) are looked up lane by lane.  A table
without its last node, or an I_0^4 with 300 more (beyond every separation here, so the
interpolants agree), takes the second."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

H = 0.67


def _inputs(nren):
    from coffe_amd import background as B
    from coffe_amd.engine import COFFE_SEP
    zb = np.linspace(0, 10, 11)
    bg = B.compute(omega_cdm=0.25, omega_baryon=0.05, h=H, bias_z=zb, s1=0.1 + 0.03 * zb, s2=0.25 - 0.01 * zb,
                   fevo1=0.5 + 0 * zb, fevo2=-0.2 + 0.05 * zb)
    bgd = dict(z=bg["z"], chi=bg["chi"], D1=bg["D1"], a=bg["a"], f=bg["f"], cH=bg["conformal_Hz"], G1=bg["G1"],
               G2=bg["G2"])
    pops = (zb, 1.2 + 0.3 * zb, 0.9 + 0.1 * zb, zb, 0.1 + 0.03 * zb, 0.25 - 0.01 * zb, 0.5 + 0 * zb, -0.2 + 0.05 * zb)
    # smooth tables on 43 small separations and a log-uniform part far past every r
    x = np.concatenate([[0.0], np.geomspace(1e-6, 0.05, 42), np.geomspace(0.1, 3e5, 700)])
    tabs = {}
    for i, (n, l) in enumerate([(0, 0), (0, 2), (0, 4), (1, 1), (1, 3), (2, 0), (2, 2), (3, 1)]):
        tabs[(n, l)] = (x, (1 + 0.3 * i) * x ** l / (1 + (x / (40 + 9 * i)) ** 2) ** (1 + l / 2 + 0.2 * i))
    chi = np.linspace(0.0, 7000.0, nren)
    div = np.concatenate([[0.0], np.geomspace(1e-4, 2e4, 296)])
    tabs[(4, 0)] = (div, 5.0 / (1 + div / 90.0))
    ren = (chi, 2.0 + np.cos(chi[:, None] / 900) * np.cos(chi[None, :] / 900))
    return bgd, pops, tabs, ren, (div, 0.5 + div / 1e4), bg


ALL = ["den", "rsd", "d1", "d2", "g1", "g2", "g3", "len", "g4", "g5"]


@pytest.mark.parametrize("flags,rule,nren", [
    (ALL, None, 101), (["len"], (1, 2, 1, 2, 1, 2), 101), (["g4"], (3, 5, 3, 7, 2, 3), 101),
    (["len", "g5"], (2, 3, 5, 13, 2, 4), 101), (ALL, (1, 3, 1, 64, 1, 2), 101), (ALL, (1, 3, 5, 13, 1, 2), 101),
    (["len", "g4", "only_cross"], (2, 8, 4, 16, 2, 4), 101), (ALL, (5, 64, 1, 5, 1, 2), 512),
    (["len", "g4", "flat_ll"], (2, 8, 4, 16, 2, 4), 400)])
def test_fetched_and_gathered(engine, flags, rule, nren):
    """both variants agree within what rounding of r^2 can move them: the terms' weights
    are regular in r there, so 1e-9 of the largest value (1e-15 times the 10^4 ... 10^6 of
    lambda^2 / r^2 at these separations)"""
    from coffe_amd.engine import integrated_corrfunc
    bgd, pops, tabs, ren, ren0, _ = _inputs(nren)
    own = dict(tabs)
    if "g4" in flags or "g5" in flags:   # also where no other table is read
        x, y = tabs[(4, 0)]
        far = np.geomspace(2.5e4, 1e6, 300)
        own[(4, 0)] = (np.concatenate([x, far]), np.concatenate([y, 5.0 / (1 + far / 90.0)]))
    own[(3, 1)] = tuple(v[:-1] for v in tabs[(3, 1)])
    own[(0, 0)] = tuple(v[:-2] for v in tabs[(0, 0)])
    zs, mus, seps = [0.7, 1.2], [-0.95, -0.2, 0.0, 0.6, 0.99], np.array([8.0, 90.0])
    print("integrated variants", flags, rule, nren, flush=True)
    out = [integrated_corrfunc(bgd, *pops, 0.30, H / 2997.92458, t, flags, zs, mus, seps, ren=ren, ren0=ren0, rule=rule)
           for t in (tabs, own)]
    for a, b in zip(*out):
        assert np.isfinite(a).all() and a.shape == (2, 5, 2)
        assert np.max(np.abs(a - b)) <= 1e-9 * np.max(np.abs(b))


@pytest.mark.parametrize("nren,n40", [(512, 512), (513, 300), (600, 513), (101, 513)])
@pytest.mark.parametrize("flags", [["g4"], ["len", "g4", "flat_ll"]])
def test_grid_and_divergent_table_sizes_vs_oracle(engine, flags, nren, n40):
    """either side of the LDS kernel's 512 nodes of I_0^4 and of the renormalisation grid, against the oracle
    on the same rule: 1e-9 of the largest value, as test_gpu_integrated.py"""
    from coffe_amd.engine import integrated_corrfunc
    from oracle import integrated as OI
    bgd, pops, tabs, ren, ren0, bg = _inputs(nren)
    div = np.concatenate([[0.0], np.geomspace(1e-4, 2e4, n40 - 1)])
    tabs[(4, 0)] = (div, 5.0 / (1 + div / 90.0))
    zs, mus, seps = [0.7, 1.2], [-0.95, 0.0, 0.6], np.array([8.0, 90.0])
    print("integrated grid sizes", flags, nren, n40, flush=True)
    _, got = integrated_corrfunc(bgd, *pops, 0.30, H / 2997.92458, tabs, flags, zs, mus, seps, ren=ren, ren0=ren0,
                                 rule=(2, 8, 4, 16, 2, 4))
    inp = OI.Inputs(tabs, bg, 0.30, H / 2997.92458, *pops, div=(*tabs[(4, 0)], 0.5 + div / 1e4), ren=ren)
    fl = {f: 1 for f in flags}
    want = np.array([[[OI.corrfunc_double(inp, fl, z, m, s, p1=2, n1=8, pu=4, nu=16) for s in seps] for m in mus] for z in zs])
    assert np.max(np.abs(got - want)) <= 1e-9 * np.max(np.abs(want))
