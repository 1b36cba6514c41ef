"""The register-held column pass (jw_regfft.hpp, k_col_reg) at every lattice size and
in every form it takes, against the other column passes and the unfused sequence."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SQRT, NOISE, FIXED, CORR = 0, 1, 3, 4


def start(jw, N):
    c = jw.Context(N)
    U = c.field()
    c.set_mv_zero_mode(1)
    c.philox(3, 1, 0)
    c.mv_init(U, 2, 1.0, 0.25, 1e-2)
    return c, U


def evolved(jw, c, U0, mode, space, coupling, mixed, steps=2):
    U = c.field()
    c.copy(U, U0)
    c.set_fused(mode)
    c.set_noise_space(space)
    c.philox(9, 2, 0)
    if mixed:
        c.evolve_mixed(U, coupling, jw.SIN_KERNEL, 1e-4, nsteps=steps)
    else:
        c.evolve(U, coupling, jw.SIN_KERNEL, 1e-4, nsteps=steps)
    out = U.download()
    U.close()
    return out


def worst(a, b):
    return np.sqrt((np.abs(a - b) ** 2).sum(axis=1)).max()


# Two correct forms of the step differ by the rounding of their transforms, which the
# kernel's N / 2 pi at the smallest momenta amplifies: 4e-12 at N = 2048 between two CPU
# implementations in FP64; the mixed form rounds to FP32 (2^29 times as coarse).
def bound(N, mixed):
    return max(1e-12, 2e-15 * N) * (2.0 ** 22 if mixed else 1.0)


@pytest.mark.parametrize("mixed", [0, 1])
@pytest.mark.parametrize("coupling", [SQRT, FIXED, CORR])
@pytest.mark.parametrize("N", [64, 128, 256, 512, 1024, 2048, 4096])
def test_position_noise_matches_unfused(jw, N, coupling, mixed):
    c, U0 = start(jw, N)
    a = evolved(jw, c, U0, jw.Context.FUSED, jw.NOISE_POSITION, coupling, mixed)
    b = evolved(jw, c, U0, jw.Context.UNFUSED, jw.NOISE_POSITION, coupling, mixed)
    assert worst(a, b) <= bound(N, mixed)
    assert worst(a, U0.download()) > 1e-3
    c.close()


@pytest.mark.parametrize("mixed", [0, 1])
@pytest.mark.parametrize("coupling", [SQRT, FIXED, CORR])
@pytest.mark.parametrize("N", [64, 128, 256, 512, 1024, 2048])
def test_momentum_noise_matches_interleaved_layout(jw, N, coupling, mixed):
    c, U0 = start(jw, N)
    a = evolved(jw, c, U0, jw.Context.FUSED, jw.NOISE_MOMENTUM, coupling, mixed)
    b = evolved(jw, c, U0, jw.Context.FUSED_INTERLEAVED, jw.NOISE_MOMENTUM, coupling, mixed)
    assert worst(a, b) <= bound(N, mixed)
    c.close()


@pytest.mark.parametrize("N,mixed", [(4096, 0), (4096, 1), (8192, 1)])
def test_large_momentum_noise_matches_narrow_strips(jw, N, mixed):
    c, U0 = start(jw, N)
    a = evolved(jw, c, U0, jw.Context.FUSED, jw.NOISE_MOMENTUM, CORR, mixed, steps=1)
    b = evolved(jw, c, U0, 8, jw.NOISE_MOMENTUM, CORR, mixed, steps=1)
    assert worst(a, b) <= bound(N, mixed)
    c.close()
