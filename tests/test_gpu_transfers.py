"""Fields into host memory, against what was written: transfers of one piece, of whole pieces
(512 KiB) and slots (2 MiB), with a remainder, and through a ring (8 slots) that comes round twice."""
import numpy as np
import pytest

import peridynamics as pd
from test_gpu_parity import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(3, 3, 3), (64, 64, 32), (61, 53, 37), (200, 200, 37)])
def test_fields_arrive_whole(need_gpu, shape):
    say("transfer", shape)
    pos, vol = pd.lattice_block(*shape, 1e-3, jitter_amplitude=0.05)
    b = pd.Body(pd.BBMaterial(), pos, vol)
    pd.material(b, horizon=1.2e-3, rho=2700.0, E=70e9)
    dh = pd.MI355XBodyDataHandler(b)
    v = np.random.default_rng(5).standard_normal((b.n_points, 3))
    dh.set("velocity", v)
    for _ in range(2):  # new arrays from a new ring, then from one in use
        assert np.array_equal(dh.get("velocity"), v)
        assert np.array_equal(dh.get("ref_position"), b.xyz)
        assert np.array_equal(dh.get("volume"), b.volume)
        assert not dh.get("damage").any()
    dh.close()


def test_condition_sources_of_listed_points(need_gpu):
    """Sets in any order and overlapping in different dimensions: every point moves with the value
    of its own source (velocity_bc! with f(t) and f(p, t))."""
    pos, vol = pd.lattice_block(9, 8, 7, 1e-3)
    b = pd.Body(pd.BBMaterial(), pos, vol)
    pd.material(b, horizon=3.015e-3, rho=2700.0, E=70e9)
    rng = np.random.default_rng(3)
    one, two = rng.permutation(b.n_points)[:90], rng.permutation(b.n_points)[:70]
    pd.point_set(b, "one", one)
    pd.point_set(b, "two", two)
    pd.velocity_bc(lambda t: 0.25, b, "one", "x")
    pd.velocity_bc(lambda p, t: 100.0 * p[0] + p[1] * t, b, "two", "y")
    dh = pd.MI355XBodyDataHandler(b)
    vv = pd.VelocityVerlet(steps=1)
    dh.init_time_solver(vv)
    dh.solve(vv)
    vh = dh.get("velocity_half")
    X = b.xyz
    assert np.array_equal(vh[one, 0], np.full(90, 0.25))
    assert np.array_equal(vh[two, 1], 100.0 * X[two, 0] + X[two, 1] * vv.dt)
    dh.close()


def test_transfers_of_several_threads(need_gpu):
    """Four threads, each with a body of its own, more than the process keeps rings for."""
    import threading
    shapes = [(64, 64, 32), (61, 53, 37), (30, 30, 30), (100, 100, 30)]
    wrong = []

    def work(k):
        pos, vol = pd.lattice_block(*shapes[k], 1e-3)
        b = pd.Body(pd.BBMaterial(), pos, vol)
        pd.material(b, horizon=1.2e-3, rho=2700.0, E=70e9)
        dh = pd.MI355XBodyDataHandler(b)
        v = np.random.default_rng(k).standard_normal((b.n_points, 3))
        dh.set("velocity", v)
        for _ in range(5):
            if not (np.array_equal(dh.get("velocity"), v) and np.array_equal(dh.get("volume"), b.volume)):
                wrong.append(k)
        dh.close()

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
