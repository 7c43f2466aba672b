"""Which bodies take packed bonds, and their bond states either way; the solution that every length of
the Krylov basis has to reach, from another preconditioner."""
import numpy as np
import pytest

import peridynamics as pd
import test_gpu_blocks
from test_gpu_nk import _env, nk_block, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["BB", "OSB"])
@pytest.mark.parametrize("horizon,points,bond_bytes", [(3.015, 32, 8), (3.015, 128, 8), (4.015, 32, 8),
                                                       (4.015, 64, 10), (5.015, 32, 10), (5.015, 64, 10)])
def test_layout_and_bond_states(need_gpu, oracle, kind, horizon, points, bond_bytes):
    """One 64-bit word holds the slot and the span of the lengths' bit patterns.  3.015 spacings: lengths
    within a factor of 4, 53 bits, and 11 bits of slot.  4.015: a little more than a factor of 4, 54
    bits, so packed with the tables of 32 points (at most 1024 entries) and not with those of 64.  5.015:
    54 bits and more than 1024 entries."""
    say("layout", kind, horizon, points)
    with _env(PDX_BLOCK_POINTS=str(points)):
        dh = pd.MI355XBodyDataHandler(test_gpu_blocks.body_of(kind, (23, 21, 12), horizon, isolated=kind == "BB", Gc=1.0))
        lay = dh.ctx.layout()
        dh.close()
        say(f"  {lay}")
        assert lay["lds_mode"] and lay["bond_bytes"] == bond_bytes
        test_gpu_blocks.test_bond_states_packed_and_not(None, oracle, kind, horizon)


@pytest.fixture(scope="module")
def solution():
    dh = pd.MI355XBodyDataHandler(nk_block(17, 17, 5))
    st = dh.solve_nk(pd.NewtonKrylov(steps=1, tol=1e-30, rel_tol=1e-9, maxiter=30, gmres_restart=20, gmres_maxiter=1000,
                                     gmres_reltol=1e-6, precond="two_level"))[0]
    u = dh.get("displacement")
    dh.close()
    assert st.residual_final < 1e-9 * st.residual_first
    return u


@pytest.mark.parametrize("restart", [30, 32, 33, 64, 65, 100])
def test_basis_lengths_reach_one_solution(need_gpu, solution, restart):
    """Relative tolerance 1e-9 on both sides, and a stiffness condition of about (17 spacings)^2."""
    say("krylov solution", restart)
    dh = pd.MI355XBodyDataHandler(nk_block(17, 17, 5))
    st = dh.solve_nk(pd.NewtonKrylov(steps=1, tol=1e-30, rel_tol=1e-9, maxiter=30, gmres_restart=restart,
                                     gmres_maxiter=1000, gmres_reltol=1e-6, precond="none"))[0]
    u = dh.get("displacement")
    dh.close()
    assert st.krylov_iters > restart
    assert np.linalg.norm(u - solution) <= 1e-6 * np.linalg.norm(solution)
