"""A batch that launches each kernel class once runs row-major planes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CORR = 4


def start(jw, N):
    c = jw.Context(N)
    U = c.field()
    c.set_mv_zero_mode(1)
    c.philox(3, 1, 0)
    c.mv_init(U, 2, 1.0, 0.25, 1e-2)
    return c, U


def worst(a, b):
    return np.sqrt((np.abs(a - b) ** 2).sum(axis=1)).max()


@pytest.mark.parametrize("mixed", [0, 1])
def test_one_launch_runs_row_major_planes_whatever_was_to_be_tuned(jw, mixed):
    """A layout left to the tuner, on a batch that launches each kernel class once."""
    b = jw.Batch([(64, 2), (128, 1)], fp32=bool(mixed))
    b.set_launch(1)
    singles = []
    for t, N in enumerate((64, 64, 128)):
        c, U = start(jw, N)
        b.set(t, U)
        c.philox(11, t, 0)
        if mixed:
            c.evolve_mixed(U, CORR, jw.SIN_KERNEL, 1e-4, nsteps=2, reunit_every=10)
        else:
            c.evolve(U, CORR, jw.SIN_KERNEL, 1e-4, nsteps=2)
        singles.append((c, U))
    for g in (0, 1):
        b.set_layout(g, -1)
    b.philox(11, 0, 0)
    b.evolve(CORR, jw.SIN_KERNEL, 1e-4, nsteps=2, reunit_every=10)
    b.sync()
    assert b.launch() == 1 and [b.layout(g) for g in (0, 1)] == [0, 0] and [b.fft_mode(g) for g in (0, 1)] == [0, 0]
    for t, (c, U) in enumerate(singles):
        got = c.field()
        b.get(t, got)
        assert worst(got.download(), U.download()) <= 1e-13 * (2.0 ** 22 if mixed else 1.0), t
    b.close()
