"""zmpm_download at the edges of its word ranges: the state just uploaded comes back in
upload order, to the bit (FP32 form: each value as the form stores it)."""
import ctypes

import numpy as np
import pytest

from ziran2020_amd import _abi as A

F32 = np.float32


def make(lib, n, precision, scenes=1, domain_nodes=64):
    rng = np.random.default_rng(n)
    dx = [1.0 / 48, 1.0 / 50, 1.0 / 53][:scenes]
    descs = [dict(dx=h, precision=precision, domain_nodes=domain_nodes) for h in dx]
    sim = A.Batch(lib, descs) if scenes > 1 else A.Simulation(lib, **descs[0])
    sim.set_materials([A.make_material(), A.make_material(A.MODEL_NEO_HOOKEAN), A.make_material(A.MODEL_NEO_HOOKEAN, fj_mixed=A.FJ_SOLID)])
    scene = rng.integers(0, scenes, n).astype(np.int32)
    st = dict(x=rng.uniform(0.3, 0.8, (n, 3)), v=rng.normal(size=(n, 3)), C=rng.normal(size=(n, 9)),
              F=np.eye(3).reshape(9) + 1e-3 * rng.normal(size=(n, 9)), m=rng.uniform(1, 2, n), V0=rng.uniform(1, 2, n),
              material=rng.integers(0, 3, n).astype(np.int32), d=rng.uniform(0, 1, n), g=rng.uniform(0, 1, n),
              plastic_state=rng.normal(size=n), J=1 + 1e-3 * rng.normal(size=n))
    sim.upload(st["x"], st["v"], st["C"], st["F"], st["m"], st["V0"], st["material"], d=st["d"], g=st["g"],
               plastic_state=st["plastic_state"], J=st["J"], scene=scene if scenes > 1 else None)
    want = dict(st)
    if precision == A.PREC_FP32:
        h = np.array(dx)[scene][:, None]
        bits = 2.0 ** (21 if domain_nodes <= 1024 else 19)
        want["x"] = np.rint(st["x"] / h * bits) * h / bits
        diag = np.eye(3).reshape(9)
        want["F"] = (st["F"] - diag).astype(F32).astype(float) + diag
        want["J"] = (st["J"] - 1).astype(F32).astype(float) + 1
        for k in ("v", "C", "m", "V0", "d", "g", "plastic_state"):
            want[k] = st[k].astype(F32).astype(float)
    return sim, want


# one particle; odd counts (two material indices a word); rows across a buffer's end; several buffers
@pytest.mark.gpu
@pytest.mark.parametrize("precision", (A.PREC_FP64, A.PREC_FP32))
@pytest.mark.parametrize("n,scenes", ((1, 1), (2, 3), (255, 1), (257, 3), (58255, 1), (131073, 2)))
def test_download_returns_the_uploaded_state(gpu, precision, n, scenes):
    sim, want = make(gpu, n, precision, scenes)
    for _ in range(2):  # the second time through the buffers already there
        out = sim.download()
        for k, w in want.items():
            assert np.array_equal(out[k], w), k
        assert not out["max_dtilde"].any()
    sim.close()


@pytest.mark.gpu
@pytest.mark.parametrize("keep", (("material",), ("F", "material", "J"), ("v", "d"), ()))
def test_download_of_some_arrays(gpu, keep):
    n = 1003
    sim, want = make(gpu, n, A.PREC_FP64)
    arrs = {k: np.full(want[k].size + 1, 7, want[k].dtype) for k in keep}  # one element more: not written
    p = A.Particles()
    p.n = n
    for k, a in arrs.items():
        setattr(p, k, a.ctypes.data_as(ctypes.POINTER(ctypes.c_int32 if k == "material" else ctypes.c_double)))
    assert sim.L.zmpm_download(sim.h, ctypes.byref(p)) == A.OK
    for k, a in arrs.items():
        assert np.array_equal(a[:-1], want[k].reshape(-1)) and a[-1] == 7, k
    sim.close()


@pytest.mark.gpu
def test_download_of_a_non_finite_position_and_a_smaller_upload(gpu):
    sim, want = make(gpu, 5000, A.PREC_FP32)
    x = want["x"][:77].copy()
    x[5, 1] = np.nan
    sim.upload(x, *(want[k][:77] for k in ("v", "C", "F", "m", "V0", "material")))
    out = sim.download(check=False)
    assert np.isnan(out["x"][5, 1]) and np.array_equal(np.delete(out["x"], 5, 0), np.delete(x, 5, 0))
    sim.close()
