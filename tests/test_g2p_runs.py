"""G2P and the damping pass where a workgroup's 256 particles span many grid blocks:
runs of one block's particles shorter than a wavefront, ending on its border, and more
runs than there are tiles staged at once (8; 4 under FLIP), against the oracle."""
import numpy as np
import pytest

from helpers import normwise, run
from ziran2020_amd import _abi as A, scenes

TOL = {A.PREC_FP64: 1e-9, A.PREC_FP32: 1e-4}  # the bars of the parity tests


def clusters(count, per, seed=3):
    """`count` clusters of `per` particles, each inside one cell and 8 nodes from the next."""
    rng = np.random.default_rng(seed)
    dx, side = 1.0 / 128, 13
    at = rng.permutation(side ** 3)[:count]
    cell = np.stack([at // side ** 2, at // side % side, at % side], 1) * 8 + 10
    n = count * per
    x = (np.repeat(cell, per, 0) + 0.6 + 0.8 * rng.random((n, 3))) * dx
    return scenes.Scene("clusters", dx, 128, 1e-4, 3, (0.0, -9.8, 0.0), [A.make_material()], [], x,
                        np.zeros(n, np.int32), np.full(n, 1000.0), np.full(n, dx ** 3 / per), scenes.identity_F(n),
                        v=rng.normal(scale=0.1, size=(n, 3)), C=rng.normal(scale=1.0, size=(n, 9)))


@pytest.mark.gpu
@pytest.mark.parametrize("precision", (A.PREC_FP64, A.PREC_FP32))
@pytest.mark.parametrize("transfer", (dict(), dict(transfer_scheme=A.FLIP_BLEND_PIC, flip_pic_ratio=0.9),
                                      dict(rpic_damping_iteration=1)))
@pytest.mark.parametrize("count,per", ((700, 1), (16, 32), (19, 28), (8, 64), (2, 257), (33, 31)))
def test_short_runs(gpu, oracle, precision, transfer, count, per):
    sc = clusters(count, per)
    g = run(gpu, sc, precision, 3, **transfer).download()
    o = run(oracle, sc, A.PREC_FP64, 3, **transfer).download()
    for k in ("x", "v", "C", "F"):
        assert normwise(g[k], o[k]) < TOL[precision], k
