"""The features of the LDS-staged kernels (several sets, surface correction, influence functions,
ZEMWan, long tables, killed points, J v, relaxation) at every block size that a large body takes.
The tests of the features have small bodies, which take blocks of 32 points; here the same tests run
with blocks of 64, 128 and 256 points, against the same oracle and tolerances."""
import inspect
import itertools

import pytest

import peridynamics as pd
import test_gpu_dr
import test_gpu_failure
import test_gpu_kernels
import test_gpu_mixed_state_based
import test_gpu_nk
import test_gpu_parity
import test_gpu_sets
import test_gpu_surface
from test_gpu_nk import _env

pytestmark = pytest.mark.gpu

TESTS = [
    test_gpu_parity.test_force_density_nonuniform_volume, test_gpu_parity.test_force_density_fp64,
    test_gpu_parity.test_force_density_cpd_zemwan, test_gpu_parity.test_mixed_force_error,
    test_gpu_parity.test_precrack_bonds, test_gpu_parity.test_stable_timestep_bit_exact,
    test_gpu_parity.test_nan_position_raises,
    test_gpu_sets.test_sets_force_fp64, test_gpu_sets.test_sets_equal_match_single_set,
    test_gpu_sets.test_sets_mixed_force, test_gpu_sets.test_sets_stable_timestep,
    test_gpu_sets.test_sets_vv_trajectory, test_gpu_sets.test_sets_dynamic_relaxation,
    test_gpu_sets.test_sets_cpd_mixed_context_runs_fp64,
    test_gpu_surface.test_box_factors_and_force, test_gpu_surface.test_sets_line_factors,
    test_gpu_surface.test_sets_with_correction_force, test_gpu_surface.test_mixed_force_with_correction,
    test_gpu_surface.test_osb_correction_with_influence_function,
    test_gpu_kernels.test_force_density, test_gpu_kernels.test_mixed_context_runs_fp64_passes,
    test_gpu_mixed_state_based.test_mixed_osb_force,
    test_gpu_mixed_state_based.test_mixed_osb_force_with_correction,
    test_gpu_mixed_state_based.test_mixed_cpd_force, test_gpu_mixed_state_based.test_cpd_models_force_fp64,
    test_gpu_failure.test_pulled_corner, test_gpu_failure.test_cpd_collinear_chain_is_killed,
    test_gpu_failure.test_tearing_bar_trajectory, test_gpu_failure.test_tearing_bar_cpd_mixed,
    test_gpu_nk.test_residual_and_jv_parity, test_gpu_nk.test_fused_jv_equals_two_force_evaluations,
    test_gpu_nk.test_preconditioners_on_a_ragged_size, test_gpu_nk.test_nk_in_mixed_context_uses_fp64_forces,
    test_gpu_dr.test_dr_materials,
]


def _cases():
    for fn in TESTS:
        axes = []
        for mark in getattr(fn, "pytestmark", []):
            if mark.name != "parametrize":
                continue
            names = [a.strip() for a in mark.args[0].split(",")]
            axes.append([dict(zip(names, v if len(names) > 1 else (v,))) for v in mark.args[1]])
        for combo in itertools.product(*axes):
            kw = {k: v for d in combo for k, v in d.items()}
            if kw.get("layout") == "global":  # has no blocks of this kind
                continue
            yield pytest.param(fn, kw, id="-".join([fn.__name__] + [getattr(v, "__name__", str(v)) for v in kw.values()]))


@pytest.mark.parametrize("points", [64, 128, 256])
@pytest.mark.parametrize("fn,kw", list(_cases()))
def test_feature(need_gpu, request, fn, kw, points):
    fixtures = {name: request.getfixturevalue(name) for name in inspect.signature(fn).parameters if name not in kw}
    with _env(PDX_BLOCK_POINTS=str(points)):
        fn(**fixtures, **kw)


@pytest.mark.parametrize("kind", ["BB", "CPD"])
def test_block_points_are_taken(need_gpu, kind):
    """A block's table has an entry per point that it reaches: the entries of all blocks fall with the
    block size.  Other values, and 256 for a correspondence body, leave the choice to the body."""
    pos, vol = pd.lattice_block(31, 30, 11, 1e-3)
    b = pd.Body({"BB": pd.BBMaterial, "CPD": pd.CMaterial}[kind](), pos, vol)
    pd.material(b, horizon=3.015e-3, rho=2700.0, E=70e9, **({} if kind == "BB" else {"nu": 0.25}))
    entries = {}
    for points in (None, 32, 64, 128, 256, 100):
        with _env(PDX_BLOCK_POINTS="" if points is None else str(points)):
            dh = pd.MI355XBodyDataHandler(b)
            entries[points] = dh.ctx.layout()["halo_entries"]
            dh.close()
    assert entries[32] > entries[64] > entries[128]
    assert entries[256] < entries[128] if kind == "BB" else entries[256] == entries[None]
    assert entries[None] == entries[100] == entries[32]
