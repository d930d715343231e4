"""zmpm_download where the runtime refuses one of its calls."""
import pytest

import hip_hooks


@pytest.mark.gpu
def test_a_refused_index_launch_is_reported(tmp_path):
    """The launch that finds each particle's place fails while other host threads take every range: an
    error, not particles in another order."""
    hip_hooks.run(tmp_path, """
        from test_download import make
        sim, want = make(gpu, 60000, A.PREC_FP32)
        p = A.Particles()
        p.n = 60000
        x, v, F = np.zeros((60000, 3)), np.zeros((60000, 3)), np.zeros((60000, 9))
        for k, a in (("x", x), ("v", v), ("F", F)):
            setattr(p, k, a.ctypes.data_as(ctypes.POINTER(ctypes.c_double)))
        hook("fail_launches").value = 1
        assert sim.L.zmpm_download(sim.h, ctypes.byref(p)) == A.E_HIP
        assert hook("fail_launches").value == 0
        out = sim.download()
        assert all(np.array_equal(out[k], want[k]) for k in ("x", "v", "F"))
        """)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", (0, 1))
@pytest.mark.parametrize("pinned", (0, 1, 2, 3))
def test_little_pinned_memory(tmp_path, precision, pinned):
    """Pinned memory for no buffer (0, 1: not even the flag, the flag alone), for one or for two: the state
    just uploaded comes back to the bit, and again once there is memory."""
    hip_hooks.run(tmp_path, """
        from test_download import make
        for n, scenes_ in ((1, 1), (60001, 2)):
            sim, want = make(gpu, n, int(sys.argv[3]), scenes_)
            for left in (int(sys.argv[4]), 1 << 30):
                hook("pinned_left").value = left
                out = sim.download()
                for k, w in want.items():
                    assert np.array_equal(out[k], w), (n, left, k)
                assert not out["max_dtilde"].any() and not out["laplacian"].any()
            p = A.Particles()
            p.n = n
            hook("pinned_left").value = int(sys.argv[4])
            assert sim.L.zmpm_download(sim.h, ctypes.byref(p)) == A.OK
            sim.close()
        """, precision, pinned)


@pytest.mark.gpu
def test_a_non_finite_position_without_pinned_memory(tmp_path):
    hip_hooks.run(tmp_path, """
        from test_download import make
        sim, want = make(gpu, 77, A.PREC_FP32)
        x = want["x"].copy()
        x[5, 1] = np.nan
        sim.upload(x, *(want[k] for k in ("v", "C", "F", "m", "V0", "material")))
        hook("pinned_left").value = 0
        out = sim.download(check=False)
        assert np.isnan(out["x"][5, 1]) and np.array_equal(np.delete(out["x"], 5, 0), np.delete(x, 5, 0))
        """)
