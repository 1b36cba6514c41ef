"""Rounding errors of the transforms and of the mixed form, held to those of the radix-8
transforms in LDS and of the site products in FP64 that earlier forms of these passes ran.
The inputs are fixed, so an error is one number; the bounds are those forms' own, on the
same inputs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CORR = 4


# rms error a mode of the unitary 2-D transform of unit white planes (variance 2 a site)
@pytest.mark.parametrize("N,lds", [(64, 3.146e-16), (256, 3.662e-16), (512, 4.087e-16), (1024, 4.318e-16),
                                   (2048, 4.516e-16), (4096, 4.902e-16)])
def test_fp64_transforms_err_no_more_than_radix_8(jw, N, lds):
    c = jw.Context(N)
    f = c.field(1)
    a = np.random.default_rng(N).normal(size=(N * N, 1, 2)).view(np.complex128)[..., 0]
    exact = a.reshape(N, N).astype(np.clongdouble)
    for dir, ref in ((1, np.fft.fft2(exact) / N), (0, np.fft.ifft2(exact) * N)):
        f.upload(a)
        c.execute2D(f, dir)
        e = np.abs(f.download().reshape(N, N) - ref)
        assert np.sqrt((e ** 2).mean()) <= 1.005 * lds
    c.close()


def mixed_error(jw, N, space, step, rows):
    """rms difference of one correlated step in the mixed form from FP64 on the same noise."""
    c = jw.Context(N)
    U0 = c.field()
    c.set_mv_zero_mode(1)
    c.philox(3, 1, 0)
    c.mv_init(U0, 2, 1.0, 0.25, 1e-2)
    out = []
    for mixed in (0, 1):
        U = c.field()
        c.copy(U, U0)
        c.set_noise_space(space)
        c.philox(9, 2, 0)
        if mixed:
            c.evolve_mixed(U, CORR, jw.SIN_KERNEL, step, nsteps=1, reunit_every=0)
        else:
            c.evolve(U, CORR, jw.SIN_KERNEL, step, nsteps=1)
        out.append(U.download()[::rows].copy())
        U.close()
    c.close()
    return np.sqrt((np.abs(out[0] - out[1]) ** 2).mean())


def test_mixed_8192_errs_no_more_than_radix_8(jw):
    assert mixed_error(jw, 8192, jw.NOISE_MOMENTUM, 1e-4, 8) <= 1.005 * 2.7275e-8


# a step this long lets the error of U xi U^dagger through: with its products in FP32 1.52e-6
def test_mixed_4096_keeps_fp64_products(jw):
    assert mixed_error(jw, 4096, jw.NOISE_POSITION, 1.0, 4) <= 1.005 * 1.4459e-6
