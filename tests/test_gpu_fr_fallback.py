"""The finite-rate residual with the surrogate's exact fallback on every node
against the residual with exact rates: the same production rates to the bit."""
import numpy as np
import pytest

from proteuscfd_amd import gpu
from proteuscfd_amd import surrogate as S
from tests.test_gpu_fr import BCT, MODEL, NE, NS, SCALES, _Mesh, load

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [gpu.PLAIN_FP64, gpu.CHOSEN_FP32])
def test_all_fallback_is_the_exact_solve(precision):
    """Temperatures on both sides of the thermo ranges' limit, compositions of every kind, so that all rate forms
    and powers of the mechanism act; then three implicit steps."""
    d = load("fr_bump_solve")
    model = MODEL.with_reference(*(float(d[k]) for k in SCALES[2:]))
    bct = np.array(BCT["fr_bump_solve"], dtype=np.int32)
    cc, net = gpu.ChemContext(model), gpu.MLP(seed=3)
    desc = S.desc(S.Transforms())
    desc.T_max = desc.T_min  # outside the box everywhere
    rng = np.random.default_rng(5)
    out = []
    for mlp in (None, net):
        f = gpu.FrContext(_Mesh(d), bct, np.tile(d["qinf"][:NE], (len(bct), 1)), cc)
        f.set_params(float(d["ref_pressure"]), float(d["ref_velocity"]), float(d["Pref"]), float(d["beta"]),
                     precision=precision, cfl=5.0, cfl_start=1.0, cfl_ramp=30, nsgs=6)
        if mlp is not None:
            f.set_surrogate(mlp, desc)
        if not out:
            q = np.tile(d["qinf"][:NE], (f.nnode + f.nbnode, 1))
            Y = rng.dirichlet(np.ones(NS), len(q))
            q[:, :NS] = q[:, :NS].sum(axis=1, keepdims=True) * Y
            q[:, NE - 1] *= rng.uniform(0.2, 1.3, len(q))  # 600 .. 3900 K
        print(f"[fr fallback] precision={precision} surrogate={mlp is not None}", flush=True)
        f.upload_q(q)
        b, norms = f.residual()
        f.upload_q(np.tile(d["qinf"][:NE], (f.nnode + f.nbnode, 1)))
        f.init_iterations()
        hist = np.array([f.step()[0] for _ in range(3)])
        if mlp is not None:
            assert f.surrogate_stats()["last_fallback"] == f.nnode
        out.append((b, norms, hist, f.download_q()[:, :NE]))
        f.close()
    for a, e in zip(out[1], out[0]):
        assert np.isfinite(a).all()
        np.testing.assert_array_equal(a, e)
    net.close()
    cc.close()
