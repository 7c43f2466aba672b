"""PDX_BB_UNROLL: bonds per lane and unrolled iteration of the bond-based step."""
import numpy as np
import pytest

import peridynamics as pd
from conftest import bond_layout
from test_gpu_blocks import body_of
from test_gpu_nk import _env
from test_gpu_parity import FP64_TOL, MIXED_TOL, displacement_field, oracle_for, say, scaled_error

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", ["lds", "lds12k", "global"])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("shape", [(13, 11, 7), (41, 40, 13)])
def test_unroll(need_gpu, oracle, shape, precision, layout):
    """Two and four bonds per iteration against the oracle.  A lane adds its FP64 bond forces one by
    one, so the numbers are the same; the mixed step of the LDS-staged layout sums an iteration's in
    FP32 first, so they are not, and its default is four."""
    say("bb unroll", shape, precision, layout)
    b = body_of("BB", shape, 3.015)
    X = b.xyz
    x = X + displacement_field(X, 3e-6)
    orc = oracle_for(oracle, b, "BB")
    orc.force(x)
    out = {}
    for unroll in ("", "2", "4"):
        with _env(PDX_BB_UNROLL=unroll), bond_layout(layout):
            dh = pd.MI355XBodyDataHandler(b, precision=precision)
            dh.set("position", x)
            dh.calc_force_density()
            out[unroll] = dh.get("b_int")
            assert scaled_error(out[unroll], orc) <= (FP64_TOL if precision == "fp64" else MIXED_TOL)
            assert np.array_equal(dh.get("n_active_bonds"), orc.n_active)
            dh.close()
    groups = precision == "mixed" and layout != "global"
    assert np.array_equal(out["2"], out["4"]) == (not groups)
    assert np.array_equal(out[""], out["4"])
