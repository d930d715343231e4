"""Scenes' start times on both sides of the 16 that travel as a kernel argument: each scene of a
batch, under a body force that depends on its own time, is the scene alone, bit for bit (FP32);
and the CFL step at the edges of the reduction's rows, against numpy."""
import numpy as np
import pytest

from ziran2020_amd import _abi as A, scenes


@pytest.mark.gpu
@pytest.mark.parametrize("count", (1, 16, 17))
def test_start_times(gpu, count):
    parts = []
    mats = [A.make_material()]
    for k in range(count):
        sc = scenes.elastic_cube(n_side_cells=2, seed=k)
        sc.materials, sc.t0, sc.body_forces = mats, 0.37 * k, [(50.0, 5.0, (1.0, 0.5, 0.0))]
        parts.append(sc)
    batch = scenes.SceneBatch("clocks", parts, 3)
    sim = batch.make(gpu, A.PREC_FP32)
    batch.run(sim, 3)
    out = sim.download()
    at = 0
    for sc in parts:
        one = sc.make(gpu, A.PREC_FP32)
        sc.run(one, 3)
        want = one.download()
        for k in ("x", "v", "C", "F"):
            assert np.array_equal(out[k][at:at + sc.n], want[k]), k
        at += sc.n


@pytest.mark.gpu
@pytest.mark.parametrize("precision", (A.PREC_FP64, A.PREC_FP32))
@pytest.mark.parametrize("n", (1, 256, 257, 65536, 65537))
def test_calculate_dt(gpu, precision, n):
    rng = np.random.default_rng(n)
    dx = 1.0 / 64
    x = rng.uniform(0.2, 0.8, (n, 3))
    v = rng.normal(size=(n, 3)).astype(np.float32).astype(float)
    sim = A.Simulation(gpu, dx=dx, precision=precision, domain_nodes=64)
    sim.set_materials([A.make_material()])
    sim.upload(x, v, np.zeros((n, 9)), scenes.identity_F(n), np.ones(n), np.ones(n), np.zeros(n, np.int32))
    for _ in range(2):
        r = sim.calculate_dt(1.0)
        speed = np.sqrt((v ** 2).sum(1)).max()
        # one rounding of each square, sum and root in the form's type
        assert abs(r["max_speed"] / speed - 1) < 4 * (2.0 ** -24 if precision == A.PREC_FP32 else 2.0 ** -53)
        assert r["dt"] == 0.6 * dx / r["max_speed"]
        step = dx / 2 ** 22 + 1e-15 if precision == A.PREC_FP32 else 0.0  # half a unit of the fixed point
        assert np.abs(r["min_corner"] - x.min(0)).max() <= step and np.abs(r["max_corner"] - x.max(0)).max() <= step
