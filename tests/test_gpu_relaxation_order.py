"""Dynamic relaxation at every block size: the adaptive damping carries the rounding of the sums from
step to step, so they keep one order, and the trajectories of all block sizes are the same numbers."""
import numpy as np
import pytest

import peridynamics as pd
from test_gpu_blocks import body_of
from test_gpu_nk import _env, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("kind", ["BB", "OSB", "CPD"])
@pytest.mark.parametrize("shape", [(9, 8, 7), (25, 25, 24), (23, 5, 3)])
def test_relaxation_is_the_same_at_every_block_size(need_gpu, kind, shape, precision):
    say("relaxation order", kind, shape, precision)
    b = body_of(kind, shape, 3.015, Gc=None)
    z = b.position[2]
    pd.point_set(b, "top", z > np.sort(z)[-shape[0]])
    pd.forcedensity_bc(lambda t: 1e7, b, "top", "z")
    out = {}
    for points in (32, 64, 128, 256):
        with _env(PDX_BLOCK_POINTS=str(points)):
            dh = pd.MI355XBodyDataHandler(b, precision=precision)
            dh.solve_dr(pd.DynamicRelaxation(steps=25))
            out[points] = [dh.get(f) for f in ("displacement", "velocity", "b_int", "n_active_bonds")]
            dh.close()
    assert np.abs(out[128][0]).max() > 0
    for points, fields in out.items():
        for a, c in zip(fields, out[128]):
            np.testing.assert_array_equal(a, c, err_msg=str(points))
