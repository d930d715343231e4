"""Particles that G2P defers, at the edges of the queues they are passed through (workgroups of
256 particles taken in turn by 16 queues): all of them yield, or one in seven, against the oracle."""
import numpy as np
import pytest

from helpers import normwise, run
from ziran2020_amd import _abi as A, scenes

TOL = {A.PREC_FP64: 1e-9, A.PREC_FP32: 1e-4}  # the bars of the parity tests


def yielding(n, every, seed=5):
    """n particles of a sheared cube; the first material yields, one particle in `every` has it."""
    rng = np.random.default_rng(seed)
    dx = 1.0 / 64
    side = int(np.ceil((n / 8) ** (1 / 3)))
    x = (16 + side * rng.random((n, 3))) * dx
    C = np.tile([0.0, 40.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0], (n, 1)) + rng.normal(scale=1.0, size=(n, 9))
    mats = [A.make_material(A.MODEL_FIXED_COROTATED, 1e4, 0.3, yield_stress=2.0, hardening=-800.0,
                            plasticity=A.PLASTICITY_VON_MISES_STVK_HENCKY), A.make_material()]
    return scenes.Scene("yielding", dx, 64, 1e-4, 3, (0.0, -9.8, 0.0), mats, [], x,
                        (np.arange(n) % every != 0).astype(np.int32), np.full(n, 1000.0), np.full(n, dx ** 3 / 8),
                        scenes.identity_F(n), v=rng.normal(scale=0.1, size=(n, 3)), C=C)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", (A.PREC_FP64, A.PREC_FP32))
@pytest.mark.parametrize("n,every", ((1, 1), (256, 1), (257, 7), (4096, 1), (4097, 1), (4353, 7), (8195, 1)))
def test_deferred_particles(gpu, oracle, precision, n, every):
    sc = yielding(n, every)
    g = run(gpu, sc, precision, 3).download()
    o = run(oracle, sc, A.PREC_FP64, 3).download()
    for k in ("x", "v", "C", "F", "plastic_state"):
        assert normwise(g[k], o[k]) < TOL[precision], k
    if n > 1:
        assert (o["plastic_state"][::every] > 2.0).any()


# deferred particles beside the next substep's page scan (a run: graphs of eight and two, an
# odd last substep) against each substep as a call of its own
@pytest.mark.gpu
@pytest.mark.parametrize("steps", (1, 2, 3, 11))
def test_run_is_its_substeps(gpu, steps):
    sc = yielding(4353, 7)
    a = run(gpu, sc, A.PREC_FP32, steps).download()
    sim = sc.make(gpu, A.PREC_FP32)
    for k in range(steps):
        sim.substep(sc.dt, sc.t0 + k * sc.dt)
    b = sim.download()
    for k in ("x", "v", "C", "F", "plastic_state"):
        assert np.array_equal(a[k], b[k]), k
