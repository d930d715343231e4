"""The list of touched super pages on both sides of one tile of flags (512 nodes per axis is the
last the page scan lists itself: 1024 flags in the float form, exactly 2048 in the double form),
with particles in the first and the last super page: the binning is the oracle's, bit for bit."""
import numpy as np
import pytest

from helpers import run
from test_large_domain import far_cubes
from ziran2020_amd import _abi as A


@pytest.mark.gpu
@pytest.mark.parametrize("domain", (64, 512, 1024))
@pytest.mark.parametrize("precision", (A.PREC_FP64, A.PREC_FP32))
def test_binning(gpu, oracle, domain, precision):
    sc = far_cubes(domain)
    for steps in (1, 4):
        g, o = run(gpu, sc, precision, steps), run(oracle, sc, precision, steps)
        gb, ob = g.binning(), o.binning()
        for k in ("keys", "order", "groups", "block_offset"):
            assert np.array_equal(gb[k], ob[k]), (steps, k)
        g.close()
