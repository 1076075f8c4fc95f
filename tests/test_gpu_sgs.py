"""The colour passes of the 5x5 SGS on graphs whose colours fall on both sides
of every dispatch rule (lanes per row, cached or streamed matrix), against the
oracle's sweep of the device's own matrix in the device's row order."""
import types

import numpy as np
import pytest

import oracle as O
from proteuscfd_amd.cases import BC_FARFIELD, Case, Params, qinf

pytestmark = pytest.mark.gpu


def ribbon(n, seed=0):
    """n nodes in a row, each joined to the next and two in three to the next
    but one: ragged rows of 1 to 4 blocks, three colours of about n/3 rows,
    the middle one with neighbours on both sides."""
    rng = np.random.default_rng(seed)
    i = np.arange(n)
    e = np.concatenate([np.stack([i[:-1], i[1:]], 1), np.stack([i[:-2], i[2:]], 1)[i[:-2] % 3 != 1]])
    e = e[np.lexsort((e[:, 1], e[:, 0]))].astype(np.int32)
    a = rng.normal(size=(len(e), 3))
    a /= np.linalg.norm(a, axis=1, keepdims=True)
    ea = np.concatenate([a, rng.uniform(0.5, 1.5, (len(e), 1))], axis=1)
    return types.SimpleNamespace(
        nnode=n, nedge=len(e), nbedge=1, edges=e.reshape(-1, 2), edge_a=ea, bedges=np.array([[0, n]], dtype=np.int32),
        bedge_a=np.array([[1.0, 0.0, 0.0, 1.0]]), bfactag=np.array([1], dtype=np.int32),
        xyz=np.stack([i, np.sin(i), np.cos(i)], 1).astype(float), vol=np.full(n, 1.0))


def pattern(m):
    """Block-CRS with every row's diagonal first, then its neighbours ascending."""
    r = np.concatenate([np.arange(m.nnode), m.edges[:, 0], m.edges[:, 1]])
    c = np.concatenate([np.arange(m.nnode), m.edges[:, 1], m.edges[:, 0]])
    o = np.lexsort((c, c != r, r))
    ia = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=m.nnode))]).astype(np.int32)
    return ia, c[o].astype(np.int32)


# rows a colour: 1 (a lone node), a ragged chunk, and about 1.6k, 6k, 60k and 140k; for each storage type the
# largest matrix does not fit the 256 MiB cache and is streamed
SIZES = [(p, n) for p in (0, 1) for n in (1, 2, 131, 5000, 20001, 180001, 420005)] + [(1, 900001)]
STREAMED = {(0, 420005), (1, 900001)}


@pytest.mark.parametrize("precision,n", SIZES)
def test_colour_passes(n, precision):
    from proteuscfd_amd import gpu
    m = ribbon(n)
    assert (2 * m.nedge * 25 * (4 if precision else 8) > 256 * 2**20) == ((precision, n) in STREAMED)
    q0 = qinf(1.4, 0.5)
    case = Case("ribbon", m, np.array([0, BC_FARFIELD], dtype=np.int32), np.tile(q0, (2, 1)), q0, Params(nsgs=3))
    print(f"[sgs] n={n} precision={precision}", flush=True)
    ctx = gpu.Context(case, Params(sorder=1, nsgs=3, precision=precision))
    rng = np.random.default_rng(1)
    q = np.tile(q0, (n + 1, 1))
    q[:, :5] *= 1.0 + 0.05 * rng.uniform(-1, 1, (n + 1, 5))
    ctx.upload_q(q)
    ctx.set_timestep(np.full(n, 0.2))
    ctx.jacobian()
    ia, ja = pattern(m)
    M = ctx.download_jacobian(ia, ja)
    b, _ = ctx.residual(it=0)
    ctx.prepare_sgs()
    order = ctx.sgs_order()
    # one sweep (no partial sums kept), several, and none
    for nsgs in (1, 3, 0):
        x, _ = ctx.sgs(nsgs)
        if nsgs == 0:
            assert not x.any()
            continue
        xo = O.sgs_on_matrix(ia, ja, ia[:-1].copy(), M, b, nsgs, order)
        # rounding of 5x5 solves on blocks dominated by vol/dt: 1e-11 / 2e-4, the bars of the mesh tests
        assert np.linalg.norm(x - xo) <= (1e-11 if precision == 0 else 2e-4) * np.linalg.norm(xo)
    ctx.close()
