"""jw_measure_corr and jw_dipole_from_corr at every size of the fused passes and beside
them, against the per-function calls and numpy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [8, 32, 64, 128, 256, 512, 1024, 2048, 4096])
def test_measure_matches_per_function_calls(jw, N):
    c = jw.Context(N)
    U = c.field()
    c.set_mv_zero_mode(1)
    c.philox(7, 1, 0)
    c.mv_init(U, 2, 1.0, 4.0, 1.0)
    corr = c.measure_corr(U)
    W, t = c.field(), c.field(1)
    c.copy(W, U)
    c.execute2D(W, 1)
    c.trace(W, t)
    c.average_and_symmetrize(t)
    ref = t.download()[:, 0].real
    # the spectra differ by the rounding of a transform, 2 log2(N^2) 2^-53 of the largest mode, the
    # trace by twice that
    assert np.abs(corr - ref).max() <= 4 * np.log2(N * N) * 2.0 ** -53 * ref.max()
    assert np.array_equal(corr, c.measure_corr(U))
    m = corr.reshape(N, N)
    f = np.roll(m[::-1], 1, 0)
    assert np.allclose(m, m.T, rtol=0, atol=1e-15 * ref.max()) and np.allclose(m, f, rtol=0, atol=1e-15 * ref.max())
    S = c.dipole_from_corr(corr)
    exact = np.fft.ifft2(m).real * (N * N) ** 2 / 3
    assert np.abs(S.reshape(N, N) - exact).max() <= 8 * np.log2(N * N) * 2.0 ** -53
    c.close()
