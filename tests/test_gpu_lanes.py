"""The edge passes on both sides of every lanes-per-node rule (four lanes up to
49,152 nodes, two above; gradient and viscous pass one above 98,304), phase by phase
against the oracle, and the fused gradient-limiter pass of the timed
iterations against the separate passes, NaN states included."""
import numpy as np
import pytest

import oracle as O
from proteuscfd_amd import cases
from proteuscfd_amd.cases import Params

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a) - b) / np.linalg.norm(b))


@pytest.mark.parametrize("kind,size", [("bump", 3), ("bump", 37), ("bump", 51), ("plate", (21, 9, 24)),
                                       ("plate", (60, 20, 45)), ("plate", (70, 27, 54))])
def test_edge_passes(kind, size):
    from proteuscfd_amd import gpu
    if kind == "bump":
        case = cases.bump_case(n=size, params=Params(sorder=2, limiter=3, cfl=5.0, nsgs=0))
    else:
        case = cases.plate_case(*size, nlayers=8, first_h=1e-2, params=Params(
            sorder=2, cfl=5.0, nsgs=0, viscous=1, reynolds=1e4, mach_ref=0.3))
    pb = O.Problem.from_case(case)
    q = pb.update_bcs(cases.perturbed_state(case, amp=0.02))
    print(f"[lanes] {kind} {size} nodes {case.mesh.nnode}", flush=True)
    ctx = gpu.Context(case)
    ctx.upload_q(q)
    ctx.reset_iteration()
    go = pb.gradient(q)
    assert rel(ctx.gradient(), go) < 1e-12
    lo = np.ones((case.mesh.nnode, 5))
    if case.params.limiter:
        lo = pb.limiter(q, go)
        assert rel(ctx.limiter(), lo) < 1e-10
        ctx.set_limiter(lo)
    bo, _ = pb.residual(q, go, lo, 1)
    b, norms = ctx.residual(it=1)
    assert rel(b, bo) < 1e-12
    assert abs(norms[0] - np.linalg.norm(bo) / bo.size) <= 1e-12 * norms[0]
    dto, _ = pb.timestep(q, 5.0)
    dt, dtmin = ctx.timestep(5.0)
    assert rel(dt, dto) < 1e-13 and dtmin == dt.min()
    ctx.close()


@pytest.mark.parametrize("limiter", [1, 2, 3])
@pytest.mark.parametrize("n,bad", [(9, None), (9, 3), (37, None), (37, 1000)])
def test_fused_pass(n, bad, limiter):
    from proteuscfd_amd import gpu
    case = cases.bump_case(n=n, params=Params(sorder=2, limiter=limiter, cfl=5.0, cfl_start=1.0, nsgs=3))
    q0 = cases.perturbed_state(case, amp=0.05)
    if bad is not None:
        q0[bad, 4] = np.nan
    print(f"[lanes] fused n={n} limiter={limiter} bad={bad}", flush=True)
    out = []
    for timing in (False, True):  # phase timing keeps gradient and limiter apart
        ctx = gpu.Context(case)
        ctx.upload_q(q0)
        ctx.reset_iteration()
        ctx.enable_phase_timing(timing)
        for _ in range(3):
            ctx.iterate()
        out.append(ctx.download_q(5))
        ctx.close()
    np.testing.assert_array_equal(np.isnan(out[0]), np.isnan(out[1]))
    # the same gradient to rounding, then FD Jacobians (h = 1e-8) on states that differ in last bits
    np.testing.assert_allclose(out[0], out[1], rtol=1e-8, atol=1e-10)
