"""The block sizes of the LDS-staged kernels against the oracle: bodies on both sides of every
size at which the points per block and the lanes per point change, ragged last blocks and
slices, isolated points, packed and unpacked bonds (the horizon decides), and the sums that
dynamic relaxation keeps in one order for every block size."""
import numpy as np
import pytest

import peridynamics as pd
from test_gpu_parity import (FP64_TOL, MIXED_TOL, bonds_equal, displacement_field, oracle_for, say,
                             scaled_error)

pytestmark = pytest.mark.gpu

# below 256 blocks of 64 points: 32 points x 16 lanes; below 160 of 128: 64 x 8; then 128 x 4
SHAPES = {"tiny": (3, 3, 3), "32x16": (37, 25, 11), "32x16 more": (31, 30, 11),
          "64x8": (32, 32, 16), "64x8 last": (40, 39, 13),
          "128x4": (41, 40, 13), "128x4 more": (61, 43, 16)}


def body_of(kind, shape, horizon, isolated=False, Gc=100.0):
    dx = 1e-3
    pos, vol = pd.lattice_block(*shape, dx, jitter_amplitude=0.05)
    if isolated:  # points without bonds, first, last and in the middle of the Morton order
        far = np.array([[-9.0, 0.0, 9.0], [-9.0, 0.5, 9.0], [-9.0, 0.0, 9.0]])
        pos = np.concatenate([pos, far], axis=1)
        vol = np.concatenate([vol, np.full(3, dx ** 3)])
    mat = {"BB": pd.BBMaterial, "OSB": pd.OSBMaterial, "CPD": pd.CMaterial}[kind]()
    b = pd.Body(mat, pos, vol)
    kw = dict(horizon=horizon * dx, rho=2700.0, E=70e9)
    if Gc is not None:
        kw["Gc"] = Gc
    if kind != "BB":
        kw["nu"] = 0.25
    pd.material(b, **kw)
    return b


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("kind", ["BB", "OSB", "CPD"])
@pytest.mark.parametrize("shape", list(SHAPES))
def test_force_density_at_block_sizes(need_gpu, oracle, kind, shape, precision):
    say("blocks", kind, shape, precision)
    if kind == "CPD" and shape == "tiny":
        pytest.skip("27 points leave single-sided correspondence neighbourhoods")
    b = body_of(kind, SHAPES[shape], 3.015)
    dh = pd.MI355XBodyDataHandler(b, precision=precision)
    orc = oracle_for(oracle, b, kind)
    bonds_equal(dh, orc)
    X = b.xyz
    x = X + displacement_field(X, 3e-6)
    dh.set("position", x)
    dh.calc_force_density()
    orc.force(x)
    assert scaled_error(dh.get("b_int"), orc) <= (FP64_TOL if precision == "fp64" else MIXED_TOL)
    assert np.array_equal(dh.get("n_active_bonds"), orc.n_active)
    dh.close()


@pytest.mark.parametrize("horizon", [3.015, 4.015, 5.015])
@pytest.mark.parametrize("kind", ["BB", "OSB"])
def test_bond_states_packed_and_not(need_gpu, oracle, kind, horizon):
    """Breaking bonds, their states and lengths with one 64-bit word per bond (3.015 spacings)
    and with separate words and lengths (the wider horizons)."""
    say("packed", kind, horizon)
    b = body_of(kind, (23, 21, 12), horizon, isolated=kind == "BB", Gc=1.0)
    dh = pd.MI355XBodyDataHandler(b)
    orc = oracle_for(oracle, b, kind)
    X = b.xyz
    m = X.shape[0] - (3 if kind == "BB" else 0)  # the isolated points stay where they are
    x = X.copy()
    x[:m] += displacement_field(X[:m], 1e-5)
    for _ in range(2):  # the second call meets the bonds that the first one broke
        dh.set("position", x)
        dh.calc_force_density()
        orc.force(x)
        act = bonds_equal(dh, orc)
        assert np.array_equal(act, orc.active)
        assert 0 < act.sum() < act.size
        assert scaled_error(dh.get("b_int"), orc) <= FP64_TOL
        x[:m] += displacement_field(X[:m, [1, 2, 0]], 5e-6)
    dh.close()


@pytest.mark.parametrize("kind", ["BB", "OSB", "CPD"])
@pytest.mark.parametrize("shape", ["32x16", "64x8"])
def test_relaxation_force_density(need_gpu, oracle, kind, shape):
    """The force density of a relaxation step, whose sums keep the order of four lanes per point
    (every group of four lanes walks the whole row), at the block sizes with more lanes."""
    say("relaxation order", kind, shape)
    b = body_of(kind, SHAPES[shape], 3.015, isolated=kind == "BB", Gc=None)
    dh = pd.MI355XBodyDataHandler(b)
    orc = oracle_for(oracle, b, kind)
    X = b.xyz
    m = X.shape[0] - (3 if kind == "BB" else 0)
    x = X.copy()
    x[:m] += displacement_field(X[:m], 3e-6)
    dh.set("position", x)
    dh.ctx.dr_init(1.0, 1.0)
    dh.ctx.dr_run(1, 1, 1.0)  # velocity_half is zero: the positions stay
    orc.force(x)
    assert scaled_error(dh.get("b_int"), orc) <= FP64_TOL
    assert np.array_equal(dh.get("n_active_bonds"), orc.n_active)
    dh.close()


@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 1, 1), (65, 1, 1), (70, 50, 40)])
def test_bond_lists_of_the_device_set_up(need_gpu, oracle, shape):
    """Bond lists, lengths and the stable time step of bodies from one point to many sort and
    scan runs, with a precrack through the larger one."""
    say("device set-up", shape)
    b = body_of("BB", shape, 3.015)
    y = b.position[1]
    if shape[1] > 1:
        pd.point_set(b, "a", (y > 0) & (y < 6e-3) & (b.position[0] < 0))
        pd.point_set(b, "b", (y <= 0) & (y > -6e-3) & (b.position[0] < 0))
        pd.precrack(b, "a", "b")
    dh = pd.MI355XBodyDataHandler(b)
    orc = oracle_for(oracle, b, "BB")
    act = bonds_equal(dh, orc)
    assert np.array_equal(act, orc.active)
    assert np.array_equal(dh.get("n_active_bonds"), orc.n_active)
    if shape[0] > 1:
        assert dh.calc_stable_timestep() == orc.stable_dt()
    dh.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("zem", ["silling", "wan"])
@pytest.mark.parametrize("horizon", [3.015, 4.015, 5.015])
def test_correspondence_failure_and_tiles(need_gpu, oracle, horizon, zem, precision):
    """Correspondence bodies whose neighbour tables fit one LDS tile (3.015 spacings) and take
    several (wider horizons), with bonds on both sides of the critical stretch: the squared
    pre-check of the failure window may not lose one."""
    say("correspondence tiles", horizon, zem, precision)
    b = body_of("CPD", (23, 21, 12), horizon, Gc=100.0)
    if zem == "wan":
        b.mat.zem = pd.ZEMWan()
    dh = pd.MI355XBodyDataHandler(b, precision=precision)
    orc = oracle_for(oracle, b, "CPD")
    X = b.xyz
    x = X + displacement_field(X, 1e-5)
    for _ in range(2):
        dh.set("position", x)
        dh.calc_force_density()
        orc.force(x)
        assert np.array_equal(dh.get("n_active_bonds"), orc.n_active)
        assert 0 < orc.n_active.sum() < dh.n_bonds
        assert scaled_error(dh.get("b_int"), orc) <= (FP64_TOL if precision == "fp64" else MIXED_TOL)
        x = x + displacement_field(X[:, [1, 2, 0]], 5e-6)
    dh.close()


@pytest.mark.parametrize("shape", ["tiny", "64x8", "128x4 more"])
def test_relaxation_steps_in_one_call(need_gpu, shape):
    """Relaxation steps of one call, where a step's update also begins the next one, equal the same
    steps in calls of their own, with time-dependent velocity and force-density conditions that
    leave out some steps (NaN)."""
    say("relaxation calls", shape)
    out = []
    for cap in (7, 1):
        b = body_of("BB", SHAPES[shape], 3.015, Gc=None)
        x = b.position[0]
        pd.point_set(b, "left", x < x.min() + 1.1e-3)
        pd.point_set(b, "right", x > x.max() - 1.1e-3)
        pd.velocity_bc(lambda t: np.nan if t == 3.0 else 1e-9 * t, b, "left", "x")
        pd.forcedensity_bc(lambda t: np.nan if t in (2.0, 5.0) else 1e5 * t, b, "right", "x")
        dh = pd.MI355XBodyDataHandler(b)
        dh.ctx.dr_init(1.0, 1.0)
        for n in range(1, 8, cap):
            dh.ctx.dr_run(n, cap, 1.0, dh.bc_values(range(n, n + cap), 1.0))
        out.append([dh.get(f) for f in ("displacement", "velocity", "velocity_half", "velocity_half_old", "b_int",
                                        "b_int_old", "b_ext", "position")])
        dh.close()
    assert np.abs(out[0][0]).max() > 0
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("kind", ["BB", "OSB"])
@pytest.mark.parametrize("shape", [(48, 37, 30), (44, 36, 30)])
def test_mixed_wide_horizon(need_gpu, oracle, kind, shape):
    """Mixed steps at 5.015 spacings in 256-point blocks (209 of them) and, where these would
    leave a quarter of the device idle (186), in 64-point ones."""
    say("mixed wide", kind, shape)
    b = body_of(kind, shape, 5.015, Gc=None)
    dh = pd.MI355XBodyDataHandler(b, precision="mixed")
    orc = oracle_for(oracle, b, kind)
    X = b.xyz
    x = X + displacement_field(X, 3e-5)
    dh.set("position", x)
    dh.calc_force_density()
    orc.force(x)
    assert scaled_error(dh.get("b_int"), orc) <= MIXED_TOL
    assert np.array_equal(dh.get("n_active_bonds"), orc.n_active)
    dh.close()
