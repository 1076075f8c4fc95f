"""Work of the library runs on non-blocking streams, which do not wait for the
null stream: device memory is cleared on the stream of the work that follows."""
import glob
import os
import re

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_no_fill_on_the_null_stream():
    """hipMemset (hipMemsetD8/D16/D32 too) takes no stream: it runs on the null one."""
    files = glob.glob(os.path.join(ROOT, "proteuscfd_amd", "csrc", "*.hip"))
    assert files
    for f in files:
        with open(f) as fh:
            code = re.sub(r"//[^\n]*", "", fh.read())
        assert not re.findall(r"\bhipMemset(?:D8|D16|D32)?\s*\(", code), f


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n", [4, 9])
def test_first_sweeps_of_a_context(n, precision):
    """The row-order correction's padding is zero from the first call on: the sweeps' norm is that of the
    correction itself, and a repeated call gives the same."""
    from proteuscfd_amd import cases, gpu
    case = cases.bump_case(n=n)
    p = cases.Params(sorder=1, nsgs=4, precision=precision)
    print(f"[fill] n={n} precision={precision}", flush=True)
    for _ in range(3):
        ctx = gpu.Context(case, p)
        ctx.upload_q(cases.perturbed_state(case, amp=0.02))
        ctx.timestep(5.0)
        ctx.jacobian()
        ctx.residual(it=0)
        ctx.prepare_sgs()
        # with one sweep there is no norm before it: delta is the correction's
        x, delta = ctx.sgs(1)
        norm = np.linalg.norm(x) / x.size
        assert abs(delta - norm) <= 1e-12 * norm
        x2, delta2 = ctx.sgs(1)
        np.testing.assert_array_equal(x2, x)
        assert delta2 == delta
        ctx.close()
