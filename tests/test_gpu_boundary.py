"""Boundary states and the boundary part of the Jacobian where half-edges of
several types meet on a node: resetting ones (noSlip, Dirichlet) before and
after characteristic ones, isothermal and adiabatic walls on one node, against
the oracle's walk in half-edge order."""
import numpy as np
import pytest

import oracle as O
from proteuscfd_amd import cases
from proteuscfd_amd.cases import (BC_DIRICHLET, BC_FARFIELD, BC_IMPERMEABLE, BC_NOSLIP, BC_SONIC_INFLOW,
                                  BC_SONIC_OUTFLOW, BC_SYMMETRY, Params)

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


# BC types of face tags 1..6 and wall temperatures (< 0 adiabatic) of tags 3 and 5
MIXES = {
    "noslip both": ([BC_FARFIELD, BC_SONIC_OUTFLOW, BC_NOSLIP, BC_SYMMETRY, BC_NOSLIP, BC_FARFIELD], -1.0, 1.1),
    "floor adiabatic": ([BC_FARFIELD, BC_FARFIELD, BC_SYMMETRY, BC_IMPERMEABLE, BC_NOSLIP, BC_SYMMETRY], 0.9, -1.0),
    "resets in between": ([BC_SONIC_INFLOW, BC_SONIC_OUTFLOW, BC_IMPERMEABLE, BC_DIRICHLET, BC_NOSLIP, BC_FARFIELD],
                          1.0, 1.0),
    "no resets": ([BC_FARFIELD, BC_SONIC_OUTFLOW, BC_IMPERMEABLE, BC_SYMMETRY, BC_IMPERMEABLE, BC_FARFIELD], 1.0, 1.0),
}


@pytest.mark.parametrize("centred", [0, 1])
@pytest.mark.parametrize("mix", list(MIXES))
def test_mixed_half_edges(mix, centred):
    types, tw3, tw5 = MIXES[mix]
    check(mix, types, {3: tw3, 5: tw5}, centred)


# Adiabatic walls whose wall-normal neighbour another half-edge resets: before (its new state is read, as in the
# walk in half-edge order) or after (its old one), in chains, and each the other's across a channel one cell wide.
# BC types of face tags 1..6, wall temperatures, cells across
RESET_NEIGHBOURS = {
    "inflow beside": ([BC_SONIC_INFLOW, BC_SONIC_OUTFLOW, BC_SYMMETRY, BC_SYMMETRY, BC_NOSLIP, BC_FARFIELD], {5: -1.0}, 4),
    "set walls beside": ([BC_DIRICHLET, BC_SONIC_OUTFLOW, BC_NOSLIP, BC_NOSLIP, BC_NOSLIP, BC_SONIC_INFLOW],
                         {3: 1.1, 4: -1.0, 5: -1.0}, 4),
    "all adiabatic": ([BC_NOSLIP, BC_NOSLIP, BC_NOSLIP, BC_NOSLIP, BC_NOSLIP, BC_NOSLIP], {}, 3),
    "thin channel": ([BC_SONIC_INFLOW, BC_SONIC_OUTFLOW, BC_NOSLIP, BC_NOSLIP, BC_NOSLIP, BC_FARFIELD],
                     {3: -1.0, 4: -1.0, 5: 0.9}, 1),
}


@pytest.mark.parametrize("centred", [0, 1])
@pytest.mark.parametrize("mix", list(RESET_NEIGHBOURS))
def test_adiabatic_wall_beside_a_reset_node(mix, centred):
    types, tw, ny = RESET_NEIGHBOURS[mix]
    check(mix, types, tw, centred, ny)


def check(mix, types, tw, centred, ny=4):
    from proteuscfd_amd import gpu
    p = Params(sorder=1, cfl=5.0, nsgs=2, viscous=1, reynolds=1.0e3, mach_ref=0.3, jac_boundary_type=centred)
    case = cases.plate_case(nx=5, ny=ny, nz=6, nlayers=2, first_h=0.05, growth=1.2, params=p)
    case.bc_type[1:7] = types
    case.twall[1:7] = -1.0
    for tag, t in tw.items():
        case.twall[tag] = t
    # distinct reference states, so that it shows which reset a half-edge saw
    for t in range(1, 7):
        case.qref[t, :5] *= 1.0 + 0.01 * t
    cases.aux(case.qref, 1.4)
    pb = O.Problem.from_case(case)
    q0 = cases.perturbed_state(case, amp=0.02)
    print(f"[boundary] {mix} centred={centred}", flush=True)
    ctx = gpu.Context(case)
    ctx.upload_q(q0)
    ctx.update_bcs()
    assert rel(ctx.download_q(5), pb.update_bcs(q0)[:, :5]) < 1e-13
    dt, _ = pb.timestep(q0, 5.0)
    ia, ja, iau, Mo, qafter = pb.jacobian(q0, dt)
    ctx.upload_q(q0)
    ctx.set_timestep(dt)
    ctx.jacobian()
    M = ctx.download_jacobian(ia, ja)
    # h = 1e-8 differences: a last bit of a flux is 1e-8 of an entry
    assert rel(M, Mo) < 1e-6 and rel(M[iau], Mo[iau]) < 1e-6
    wall = np.unique(case.mesh.bedges[np.isin(np.asarray(types)[case.mesh.bfactag - 1], BC_NOSLIP), 0])
    for i in wall:  # the hard-set sub-rows exactly
        rows = slice(ia[i], ia[i + 1])
        np.testing.assert_array_equal(M[rows][:, 1:4], Mo[rows][:, 1:4])
        np.testing.assert_allclose(M[rows][:, 4], Mo[rows][:, 4], rtol=0, atol=1e-14)
    assert rel(ctx.download_q(5), qafter[:, :5]) < 1e-13
    ctx.close()
