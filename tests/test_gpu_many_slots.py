"""Bodies of more than 2^32 bond slots: the kernels over the slots may not need a thread for each."""
import numpy as np
import pytest

import peridynamics as pd
from conftest import bond_layout
from peridynamics import _lib
from test_gpu_parity import FP64_TOL, MIXED_TOL, say

pytestmark = pytest.mark.gpu

DX = 1e-3


@pytest.mark.parametrize("precision,layout,shape,horizon,bond_bytes",
                         [("fp64", "lds", (256, 256, 272), 3.9, 8),
                          ("mixed", "global", (256, 144, 136), 6.015, 12)])
def test_more_than_2_to_32_slots(need_gpu, precision, layout, shape, horizon, bond_bytes):
    """Packed bonds (17.8 M points, 250 bonds each) and the FP32 lengths of the global-gather layout
    (5 M points, 924 bonds each): all bonds are found, and a stretched body's force density agrees
    with its definition at both ends of the slots, at corners and at points between."""
    say("slots", precision, layout, shape)
    X = DX * np.indices(shape, dtype=np.float64).reshape(3, -1).T
    n = X.shape[0]
    r = int(horizon)
    o = np.array([(i, j, k) for i in range(-r, r + 1) for j in range(-r, r + 1) for k in range(-r, r + 1)
                  if 0 < i * i + j * j + k * k <= horizon ** 2])
    p = pd.materials.get_point_params(pd.BBMaterial(), dict(horizon=horizon * DX, rho=2700.0, E=70e9))
    q = _lib.PdxParams()
    for name in ("delta", "rho", "bc", "epsc"):
        setattr(q, name, getattr(p, name))
    with bond_layout(layout):
        ctx = _lib.Context(precision=_lib.PDX_FP64 if precision == "fp64" else _lib.PDX_MIXED)
        ctx.set_points(X, DX ** 3, np.zeros(n, np.uint8))
        ctx.set_material(_lib.PDX_BB, q)
        nb = ctx.build_bonds()
    lay = ctx.layout()
    say(f"  {n} points, {nb} bonds, {lay}")
    assert nb == sum(int(np.prod([shape[d] - abs(int(v[d])) for d in range(3)])) for v in o)
    assert lay["bond_slots"] > 2 ** 32 and lay["bond_bytes"] == bond_bytes
    F = np.eye(3) + 1e-2 * np.array([[1.0, 0.3, 0.0], [0.2, -0.5, 0.1], [0.0, 0.4, 0.7]])
    x = X @ F.T
    ctx.set_field("position", x)
    ctx.force_density()
    b, na = ctx.get_field("b_int"), ctx.get_field("n_active_bonds")
    ctx.close()
    assert int(na.sum()) == nb
    at = np.concatenate([[0, n - 1], np.ravel_multi_index(np.array([(0, -1, 0), (-1, 0, -1)]).T % np.array(shape)[:, None], shape),
                         np.random.default_rng(4).integers(0, n, 60)])
    for i in at:
        c = np.array(np.unravel_index(i, shape)) + o
        j = np.ravel_multi_index(c[np.all((c >= 0) & (c < shape), axis=1)].T, shape)
        D, d = X[j] - X[i], x[j] - x[i]
        L, l = np.linalg.norm(D, axis=1), np.linalg.norm(d, axis=1)
        t = p.bc * (l - L) / L * DX ** 3
        assert na[i] == len(j)
        err = np.abs(b[i] - (t / l) @ d).max() / np.abs(t).sum()
        assert err <= (FP64_TOL if precision == "fp64" else MIXED_TOL)
