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
