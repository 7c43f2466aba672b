"""The norm of v inside J v: its partial sums are added in one order whatever the workgroup that
adds them, so the perturbation of the one-kernel J v is that of two force evaluations."""
import numpy as np
import pytest

import peridynamics as pd
from test_gpu_nk import _env, nk_block, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("shape", [(13, 11, 7), (40, 36, 33)])
def test_norm_order_is_that_of_two_force_evaluations(need_gpu, shape, precision):
    """12 and 557 partial sums (one per 256 dofs): the same bits from every form of J v.  A step of
    ||v||^2 in its last place moves the perturbation, and with it every component of J v."""
    say("nk norm order", shape, precision)
    b = nk_block(*shape)
    rng = np.random.default_rng(12)
    u = 1e-7 * rng.standard_normal((b.n_points, 3))
    vs = [rng.standard_normal((b.n_points, 3)) * 10.0 ** rng.uniform(-2, 2, (b.n_points, 1)) for _ in range(8)]
    out = {}
    for name, env in (("one pass", {}), ("sequential", {"PDX_JV_ONE_PASS": "0"}),
                      ("two kernels", {"PDX_JV_TWO_KERNELS": "1"})):
        with _env(**env):
            dh = pd.MI355XBodyDataHandler(b, precision=precision)
            dh.init_newton_krylov(pd.NewtonKrylov(steps=1))
            dh.set("displacement", u)
            dh.set("position", b.xyz + u)
            out[name] = [dh.ctx.jv(v) for v in vs]
            dh.close()
    for name in ("one pass", "sequential"):
        for a, c in zip(out[name], out["two kernels"]):
            assert np.all(np.isfinite(a)) and np.max(np.abs(a)) > 0
            np.testing.assert_array_equal(a, c, err_msg=name)
