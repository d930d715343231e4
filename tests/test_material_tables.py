"""Material tables on both sides of the 16 records that G2P stages in LDS, and of the 64-bit words of
P2G's table of the materials that carry the phase field: every third material does, the particles
are spread over all of them, against the oracle."""
import numpy as np
import pytest

from helpers import normwise
from ziran2020_amd import _abi as A, scenes

TOL = {A.PREC_FP64: 1e-9, A.PREC_FP32: 1e-4}  # the bars of the parity tests


@pytest.mark.gpu
@pytest.mark.parametrize("precision", (A.PREC_FP64, A.PREC_FP32))
@pytest.mark.parametrize("transfer", (dict(), dict(transfer_scheme=A.FLIP_BLEND_PIC, flip_pic_ratio=0.9)))
@pytest.mark.parametrize("count", (1, 16, 17, 65, 256))
def test_tables(gpu, oracle, precision, transfer, count):
    sc = scenes.damage_slab(n=3000, dx=1.0 / 32, domain_nodes=64, sigma_crit=20.0)
    mats = []
    for k in range(count):
        E = 1e4 * (1 + k / 256)
        mats.append(A.make_material(A.MODEL_QR_STABLE_NEO_HOOKEAN, E, 0.3, has_damage=True, directors=((1, 0, 0),),
                                    alphas=(-0.9,), residual_phase=0.001, l0=2 * sc.dx, sigma_crit=20.0 + k, eta=0.1, zeta=1.0)
                    if k % 3 == 0 else A.make_material(A.MODEL_NEO_HOOKEAN, E, 0.3))
    sc.materials = mats
    rng = np.random.default_rng(count)
    sc.material = (np.arange(sc.n) % count).astype(np.int32)
    sc.C = rng.normal(scale=2.0, size=(sc.n, 9))
    d = rng.uniform(0, 0.5, sc.n)  # also on the particles whose materials ignore it
    out = []
    for lib, prec in ((gpu, precision), (oracle, A.PREC_FP64)):
        sim = sc.make(lib, prec, **transfer)
        sim.upload(sc.x, sc.v, sc.C, sc.F, sc.m, sc.V0, sc.material, d=d, g=(1 - d) ** 2)
        sc.run(sim, 5)
        out.append(sim.download())
    for k in ("x", "v", "C", "F"):
        assert normwise(out[0][k], out[1][k]) < TOL[precision], k
    assert normwise(out[0]["d"], out[1]["d"]) < 10 * TOL[precision]
