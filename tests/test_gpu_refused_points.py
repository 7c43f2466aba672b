"""Points that pdx_set_points refuses never reach the device."""
import numpy as np
import pytest

import peridynamics as pd
from peridynamics import _lib
from test_gpu_parity import say

pytestmark = pytest.mark.gpu


def _material(ctx):
    p = pd.materials.get_point_params(pd.BBMaterial(), dict(horizon=3.015e-3, rho=2700.0, E=70e9))
    q = _lib.PdxParams()
    for name, value in (("delta", p.delta), ("rho", p.rho), ("bc", p.bc), ("epsc", p.epsc)):
        setattr(q, name, value)
    ctx.set_material(_lib.PDX_BB, q)


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("at", [0, 200, -1])
def test_non_finite_positions(need_gpu, bad, at):
    """A context whose only points were refused has none to build; one that held a body keeps it."""
    say("refused points", bad, at)
    pos, vol = pd.lattice_block(6, 7, 8, 1e-3)
    X = np.ascontiguousarray(pos.T)
    wrong = np.concatenate([X, X[:5] + 1.0])
    wrong.reshape(-1)[at] = bad
    ctx = _lib.Context()
    _material(ctx)
    with pytest.raises(_lib.ArgumentError, match="non-finite position"):
        ctx.set_points(wrong, 1e-9)
    with pytest.raises(_lib.PdxError, match="pdx_set_points first"):
        ctx.build_bonds()
    ctx.set_points(X, vol)
    nb = ctx.build_bonds()
    with pytest.raises(_lib.ArgumentError, match="non-finite position"):
        ctx.set_points(wrong, 1e-9)
    assert np.array_equal(ctx.get_field("ref_position"), X)
    assert ctx.build_bonds() == nb > 0  # the bonds again, from the points that are there
    ctx.close()


def test_extent_beyond_the_numbers(need_gpu):
    """Finite positions whose extent is not: refused before anything is counted or launched."""
    ctx = _lib.Context()
    _material(ctx)
    ctx.set_points(np.array([[-1.5e308, 0, 0], [1.5e308, 0, 0]]), 1e-9)
    with pytest.raises(_lib.PdxError, match="extent"):
        ctx.build_bonds()
    ctx.close()
