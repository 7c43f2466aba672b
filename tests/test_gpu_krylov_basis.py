"""The Gram-Schmidt kernels over the lengths of the Krylov basis at which they change: up to 32
vectors in registers, up to 64, and longer; and a vector whose last block is partly empty."""
import numpy as np
import pytest

import peridynamics as pd
from test_gpu_nk import nk_block, say

pytestmark = pytest.mark.gpu

_SOLVED = {}


@pytest.mark.parametrize("restart", [30, 32, 33, 64, 65, 100])
def test_basis_lengths(need_gpu, restart):
    """Every restart length reaches the relative tolerance 1e-9 and the same displacement: its error
    is the tolerance times the condition of the stiffness, about (17 spacings)^2, so 1e-6."""
    say("krylov basis", restart)
    b = nk_block(17, 17, 5)
    nk = pd.NewtonKrylov(steps=1, tol=1e-30, rel_tol=1e-9, maxiter=30, gmres_restart=restart,
                         gmres_maxiter=1000, gmres_reltol=1e-6, precond="none")
    dh = pd.MI355XBodyDataHandler(b)
    st = dh.solve_nk(nk)[0]
    u = dh.get("displacement")
    dh.close()
    say(f"  newton {st.newton_iters} krylov {st.krylov_iters}")
    assert st.krylov_iters > restart  # at least one full cycle
    assert st.residual_final < 1e-9 * st.residual_first
    ref = _SOLVED.setdefault("u", u)
    assert np.linalg.norm(u - ref) <= 1e-6 * np.linalg.norm(ref)
