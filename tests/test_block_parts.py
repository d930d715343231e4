"""P2G of blocks that several workgroups share, and of blocks at the sizes where the in-block order
changes its stage (1792 | 4504 particles in the float form, 1296 | 6416 in the double form) or a part
gains a chunk of 128: against the oracle, and in the float form bit for bit against one workgroup
that takes all blocks in turn."""
import numpy as np
import pytest

from helpers import normwise
from ziran2020_amd import _abi as A, scenes

TOL = {A.PREC_FP64: 1e-9, A.PREC_FP32: 1e-4}  # the bars of the parity tests


def crowded(n, seed=11):
    """n particles in one grid block, and 40 in another."""
    rng = np.random.default_rng(seed)
    dx = 1.0 / 64
    x = np.concatenate([16.6 + rng.random((n, 3)) * (1.8, 3.8, 3.8), 28.6 + rng.random((40, 3))]) * dx
    m = n + 40
    return scenes.Scene("crowded", dx, 64, 1e-4, 3, (0.0, -9.8, 0.0), [A.make_material()], [], x,
                        np.zeros(m, np.int32), np.full(m, 1000.0), np.full(m, 32 * dx ** 3 / m), scenes.identity_F(m),
                        v=rng.normal(scale=0.1, size=(m, 3)), C=rng.normal(scale=1.0, size=(m, 9)))


@pytest.mark.gpu
@pytest.mark.parametrize("precision", (A.PREC_FP64, A.PREC_FP32))
@pytest.mark.parametrize("transfer", (dict(), dict(mls_mpm=True), dict(rpic_damping_iteration=1)))
@pytest.mark.parametrize("n", (1, 128, 129, 1024, 1025, 1297, 1793, 4504, 4505, 6417))
def test_parts(gpu, oracle, precision, transfer, n):
    sc = crowded(n)
    out = []
    for lib, prec, wgs in ((gpu, precision, 0), (gpu, precision, 1), (oracle, A.PREC_FP64, 0)):
        sim = sc.make(lib, prec, **transfer)
        if wgs:
            sim.set_launch_config(p2g_wgs=wgs)
        sc.run(sim, 3)
        out.append(sim.download())
    for k in ("x", "v", "C", "F"):
        assert normwise(out[0][k], out[2][k]) < TOL[precision], k
        assert normwise(out[1][k], out[2][k]) < TOL[precision], k
        assert precision == A.PREC_FP64 or np.array_equal(out[0][k], out[1][k]), k


def grid_blocks(sc):
    """The float form's 4x4x4-node blocks that the particles' stencils may reach."""
    b = np.unique(np.floor(sc.x / sc.dx - 0.5).astype(int) // 4, axis=0)
    halo = np.stack(np.meshgrid(*[(0, 1)] * 3, indexing="ij"), -1).reshape(-1, 1, 3)
    return len(np.unique((b + halo).reshape(-1, 3), axis=0))


@pytest.mark.gpu
@pytest.mark.parametrize("variant", range(16))
@pytest.mark.parametrize("share", (8, 2, 1))
def test_parts_in_every_variant(gpu, variant, share):
    """Every compiled variant where each block has workgroups of its own: eight (the default), two and one,
    with some left over and in no multiple of the XCDs."""
    sc = scenes.damage_slab(n=8000, dx=1 / 64, size=(0.5, 0.15, 0.15), domain_nodes=128, sigma_crit=20.0, pull_speed=0.5)
    blocks = grid_blocks(sc)
    assert 200 < blocks < 2048 // 8
    one, sim = sc.make(gpu, A.PREC_FP32), sc.make(gpu, A.PREC_FP32)
    one.set_launch_config(p2g_wgs=1, variant=0)
    sim.set_launch_config(variant=variant, **({} if share == 8 else dict(p2g_wgs=share * blocks + blocks // 4 | 1)))
    out = []
    for s in (one, sim):
        sc.run(s, 4)
        out.append(s.download())
    for k in ("x", "v", "C", "F", "d", "g"):
        assert np.array_equal(out[0][k], out[1][k]), k
    assert out[0]["d"].max() > 0
