"""What is not finite in a field stays visible: every mode of its plane, and no other plane."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("N", [32, 64, 128, 512, 1024, 2048])
def test_transform_of_a_plane_with_one_bad_site(jw, N, bad):
    c = jw.Context(N)
    a = np.random.default_rng(N).normal(size=(N * N, 9, 2)).view(np.complex128)[..., 0]
    f = c.field(9, a)
    for dir in (1, 0):
        f.upload(a)
        c.execute2D(f, dir)
        clean = f.download()
        b = a.copy()
        b[N * (N // 3) + 5, 4] = bad
        f.upload(b)
        c.execute2D(f, dir)
        got = f.download()
        assert not np.isfinite(got[:, 4]).any()
        rest = [k for k in range(9) if k != 4]
        assert np.array_equal(got[:, rest], clean[:, rest])
    c.close()


@pytest.mark.parametrize("mixed", [0, 1])
@pytest.mark.parametrize("N", [64, 512])
def test_a_bad_site_spoils_the_measurement_and_the_step(jw, N, mixed):
    c = jw.Context(N)
    U = c.field()
    c.set_unit(U)
    a = U.download()
    a[7, 0] = np.nan
    U.upload(a)
    assert not np.isfinite(c.measure_corr(U)).any()
    c.philox(1, 0, 0)
    if mixed:
        c.evolve_mixed(U, 3, jw.SIN_KERNEL, 1e-4, nsteps=1)
    else:
        c.evolve(U, 3, jw.SIN_KERNEL, 1e-4, nsteps=1)
    assert np.isnan(U.download()).any(axis=1).all()
    c.close()
