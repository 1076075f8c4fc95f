"""Rates, source and source Jacobian of made-up mechanisms whose exponents take
every branch of the mass-action and Arrhenius powers, for the species counts
with and without a compiled form, against the oracle."""
import numpy as np
import pytest

import oracle as O
from proteuscfd_amd import chem

pytestmark = pytest.mark.gpu

AIR = chem.load_air5()


def mechanism(ns, seed):
    """ns species (a tenth of air's thermo, so that the equilibrium constants' exponents stay below about 10: an
    exponent x rounds to x eps, which a forward difference multiplies by 1e8), two reactions of each rate form
    with reactant and product powers 0, 1, 2, 3, 1/2 and Arrhenius powers
    -1.5 .. 1.5 and 0.7."""
    rng = np.random.default_rng(seed)
    nr = 8
    pick = np.arange(ns) % AIR.ns
    loc = -np.ones((nr, chem.MAXLOC), dtype=np.int32)
    nup, nupp, eff = np.zeros((nr, chem.MAXLOC)), np.zeros((nr, chem.MAXLOC)), np.ones((nr, chem.MAXLOC))
    nloc = np.zeros(nr, dtype=np.int32)
    for r in range(nr):
        k = int(rng.integers(min(2, ns), ns + 1))
        nloc[r] = k
        loc[r, :k] = rng.permutation(ns)[:k]
        nup[r, :k] = rng.choice([0.0, 1.0, 2.0, 3.0, 0.5], k)
        nupp[r, :k] = rng.choice([0.0, 1.0, 2.0, 3.0], k)
        eff[r, :k] = rng.choice([1.0, 2.5, 9.0], k)
    return chem.ChemModel(
        symbols=[f"S{i}" for i in range(ns)], mw=AIR.mw[pick] * (1 + 0.01 * np.arange(ns)), lo=0.1 * AIR.lo[pick],
        hi=0.1 * AIR.hi[pick], rtype=np.arange(nr, dtype=np.int32) % 4, tb=(np.arange(nr, dtype=np.int32) // 2) % 2,
        A=10.0 ** rng.uniform(0, 4, nr), EA=rng.uniform(100.0, 4000.0, nr),
        n=np.array([0.0, 1.0, -1.0, 0.5, -0.5, 1.5, -1.5, 0.7]), nloc=nloc, loc=loc, nup=nup, nupp=nupp, eff=eff,
        ref_density=0.9, ref_time=2e-3, ref_temperature=300.0)


@pytest.mark.parametrize("ns", [1, 3, 5, 8])
@pytest.mark.parametrize("n", [1, 63, 200])
def test_exponents(ns, n):
    from proteuscfd_amd import gpu
    m = mechanism(ns, 10 * ns)
    rng = np.random.default_rng(n)
    T = rng.uniform(400.0, 4000.0, n)
    rhoi = rng.uniform(0.01, 1.0, (n, ns))
    rhoi[0, 0] = 0.0  # 0 ** 0 = 1
    print(f"[chem] exponents ns={ns} n={n}", flush=True)
    ctx, oc = gpu.ChemContext(m), O.Chem(m)
    w = ctx.wdot(rhoi, T)
    q = np.concatenate([rhoi / m.ref_density, rng.uniform(-1, 1, (n, 3)), (T / m.ref_temperature)[:, None]], axis=1)
    vol = rng.uniform(0.5, 2.0, n)
    s, J = ctx.source(q, vol)
    np.testing.assert_array_equal(ctx.source(q, vol, jacobian=False), s)
    for i in range(n):
        wo = oc.wdot(rhoi[i], T[i])
        sc = max(np.abs(wo).max(), 1e-300)
        # sums of signed terms that are each good to a few ulp of exp(EA/T) and the powers
        assert np.abs(w[i] - wo).max() <= 1e-12 * sc, (i, w[i], wo)
        so, Jo = oc.source(q[i], vol[i]), oc.source_jacobian(q[i], vol[i])
        ss = max(np.abs(so).max(), 1e-300)
        assert np.abs(s[i] - so).max() <= 1e-12 * ss
        # forward differences: 1e-6 of the block plus the source's rounding over h = 1e-8
        assert np.abs(J[i] - Jo).max() <= 1e-6 * np.abs(Jo).max() + 1e-14 * ss / 1e-8
    ctx.close()
