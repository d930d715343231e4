"""zmpm_calculate_dt without pinned memory for its rows."""
import pytest

import hip_hooks


@pytest.mark.gpu
@pytest.mark.parametrize("precision", (0, 1))
@pytest.mark.parametrize("n", (1, 257, 65537))
def test_without_pinned_memory(tmp_path, precision, n):
    """The step, speed and corners of the device rows are those of the pinned ones, to the bit."""
    hip_hooks.run(tmp_path, """
        from test_download import make
        sim, want = make(gpu, int(sys.argv[4]), int(sys.argv[3]))
        out = []
        for left in (0, 1 << 30):
            hook("pinned_left").value = left
            out.append(sim.calculate_dt(1.0))
        assert out[0].keys() == out[1].keys()
        for k in out[0]:
            assert np.array_equal(out[0][k], out[1][k]), k
        assert abs(out[0]["max_speed"] / np.sqrt((want["v"] ** 2).sum(1)).max() - 1) < 1e-6
        """, precision, n)
