"""pdx_build_bonds again after a build that was refused half way."""
import numpy as np
import pytest

import peridynamics as pd
from peridynamics import _lib
from test_gpu_parity import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("shape", [(3, 3, 3), (13, 11, 7), (41, 40, 13)])
def test_refused_then_wider(need_gpu, shape, precision):
    """The surface correction refuses a correspondence body when its bonds and tables are on the
    device.  Without it and with a wider horizon (and with a narrower one after that) the context
    gives the bonds, tables and memory of one that never failed."""
    say("rebuild", shape, precision)
    pos, vol = pd.lattice_block(*shape, 1e-3, jitter_amplitude=0.05)
    X = np.ascontiguousarray(pos.T)

    def params(horizon):
        p = pd.materials.get_point_params(pd.CMaterial(), dict(horizon=horizon * 1e-3, rho=2700.0, E=70e9, nu=0.25))
        q = _lib.PdxParams()
        for name in ("delta", "rho", "E", "nu", "G", "K", "bc", "epsc", "mu"):
            setattr(q, name, getattr(p, name))
        q.lambda_ = p.lam
        q.zem_cs, q.maxdmg = 100.0, 0.85
        return q

    def context():
        ctx = _lib.Context(precision=_lib.PDX_FP64 if precision == "fp64" else _lib.PDX_MIXED)
        ctx.set_points(X, vol)
        return ctx

    def state(ctx):
        return (*ctx.get_bonds(), ctx.layout(), ctx.info())

    again = context()
    again.set_material(_lib.PDX_CPD, params(2.015))
    again.set_surface_correction(1)
    with pytest.raises(_lib.PdxError, match="EnergySurfaceCorrection"):
        again.build_bonds()
    again.set_surface_correction(0)
    for horizon in (4.015, 3.015):
        again.set_material(_lib.PDX_CPD, params(horizon))
        again.build_bonds()
        fresh = context()
        fresh.set_material(_lib.PDX_CPD, params(horizon))
        fresh.build_bonds()
        for a, f in zip(state(again), state(fresh)):
            assert np.array_equal(a, f) if isinstance(a, np.ndarray) else a == f
        fresh.close()
    again.close()
