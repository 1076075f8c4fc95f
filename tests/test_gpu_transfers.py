"""Callers' arrays to and from the device's component arrays: every row width, below and above the size up to which
they go through pinned memory (262144 values), bit for bit."""
import numpy as np
import pytest

from proteuscfd_amd.cases import Params, bump_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [4, 24, 27, 30])
@pytest.mark.parametrize("nvars", [5, 6, 10, 13])
def test_state_round_trip(n, nvars):
    from proteuscfd_amd import gpu

    c = bump_case(n=n)
    ntot = c.mesh.nnode + len(c.mesh.bedges)
    print(f"[transfers] n={n} nvars={nvars} values={5 * ntot}", flush=True)
    ctx = gpu.Context(c, Params(sorder=2, limiter=0, nsgs=0))
    rng = np.random.default_rng(n)
    q = rng.uniform(0.5, 1.5, (ntot, nvars))
    q[:, 4] += 4.0
    ctx.upload_q(q)
    out = np.full((ntot, nvars), -7.0)
    assert gpu.lib().pcfd_download_q(ctx.h, gpu._d(out), nvars) == 0
    np.testing.assert_array_equal(out[:, :5], q[:, :5])
    if nvars < 10:
        np.testing.assert_array_equal(out[:, 5:], -7.0)
        return
    rho, g, gm1 = q[:, 0], 1.4, 1.4 - 1.0
    u, v, w = q[:, 1] / rho, q[:, 2] / rho, q[:, 3] / rho
    v2h = 0.5 * (u * u + v * v + w * w)
    P = gm1 * (q[:, 4] - 0.5 * rho * (u * u + v * v + w * w))
    T = g * (gm1 * (q[:, 4] - rho * v2h)) / rho
    np.testing.assert_array_equal(out[:, 5:10], np.stack([T, P, u, v, w], axis=1))
    np.testing.assert_array_equal(out[:, 10:], -7.0)


@pytest.mark.parametrize("n", [4, 24, 40])
def test_time_step_and_limiter_round_trip(n):
    from proteuscfd_amd import gpu

    c = bump_case(n=n)
    nn = c.mesh.nnode
    print(f"[transfers] n={n} nodes={nn}", flush=True)
    ctx = gpu.Context(c, Params(sorder=2, limiter=1, cfl=5.0, nsgs=0))
    ctx.upload_q(c.initial_state()[:, :5])
    ctx.reset_iteration()
    dt, dtmin = ctx.timestep(5.0)
    assert dt.shape == (nn,) and (dt > 0).all() and dtmin == dt.min()
    lim = ctx.limiter()
    assert lim.shape == (nn, 5) and ((lim >= 0) & (lim <= 1 + 1e-12)).all()
    b, norms = ctx.residual(it=2)
    # a sum of 5 nn squares in another order: nn * eps relative
    np.testing.assert_allclose(norms[0], np.sqrt((b * b).sum()) / (5 * nn), rtol=5 * nn * 2.3e-16, atol=1e-30)
    np.testing.assert_allclose(norms[1:], np.sqrt((b * b).sum(0)) / nn, rtol=5 * nn * 2.3e-16, atol=1e-30)
