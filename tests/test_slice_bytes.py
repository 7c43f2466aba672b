"""The slice pointers in the byte formula of the bond-based step."""
import os
import sys

import pytest

import peridynamics as pd
from conftest import ROOT, bond_layout

sys.path.insert(0, ROOT)
import bench  # noqa: E402


@pytest.mark.parametrize("points", [64, 16, 8, 4])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 1000])
def test_slices_of_the_layout(n, points):
    lay = {"lds_mode": True, "halo_entries": 100, "bond_bytes": 8, "slice_points": points}
    pointers = 8 * -(-n // points)
    assert bench.step_bytes(n, 5000, "fp64", lay)[0] == 8 * 5000 + 168 * n + pointers + 400
    assert bench.step_bytes(n, 5000, "mixed", lay)[0] == 2 * 5000 + 200 * n + pointers + 400


@pytest.mark.gpu
@pytest.mark.parametrize("layout,block,points", [("lds", 32, 4), ("lds", 64, 8), ("lds", 128, 16), ("lds", 256, 16),
                                                 ("global", 128, 64)])
def test_layout_names_its_slices(need_gpu, layout, block, points):
    pos, vol = pd.lattice_block(9, 8, 7, 1e-3)
    b = pd.Body(pd.BBMaterial(), pos, vol)
    pd.material(b, horizon=3.015e-3, rho=2700.0, E=70e9)
    old = os.environ.get("PDX_BLOCK_POINTS")
    os.environ["PDX_BLOCK_POINTS"] = str(block)
    try:
        with bond_layout(layout):
            dh = pd.MI355XBodyDataHandler(b)
    finally:
        os.environ.pop("PDX_BLOCK_POINTS")
        if old is not None:
            os.environ["PDX_BLOCK_POINTS"] = old
    assert dh.ctx.layout()["slice_points"] == points
    dh.close()
