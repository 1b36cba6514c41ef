"""One launch per kernel class over every lattice size of a batch, on a batch's first
evolution: the coupling tables are built on the groups' own streams and have to be
whole before the launch on the batch's stream reads them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SQRT, FIXED, CORR = 0, 3, 4


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
@pytest.mark.parametrize("coupling,space", [(SQRT, 0), (SQRT, 1), (FIXED, 0), (FIXED, 1), (CORR, 0), (CORR, 1)])
def test_one_launch_batch_matches_single_lattices(jw, coupling, space, mixed):
    """Every size side by side in one launch: several strips of a small size in one workgroup."""
    groups = [(64, 3), (128, 2), (256, 2), (512, 1), (1024, 1), (2048, 1)]
    b = jw.Batch(groups, fp32=bool(mixed))
    b.set_noise_space(space)
    for g in range(len(groups)):
        b.set_layout(g, 0)
    b.set_launch(1)
    singles, t = [], 0
    for N, count in groups:
        c, U0 = start(jw, N)
        for _ in range(count):
            b.set(t, U0)
            U = c.field()
            c.copy(U, U0)
            c.set_noise_space(space)
            c.philox(11, t, 0)
            if mixed:
                c.evolve_mixed(U, coupling, jw.SIN_KERNEL, 1e-4, nsteps=2, reunit_every=10)
            else:
                c.evolve(U, coupling, jw.SIN_KERNEL, 1e-4, nsteps=2)
            singles.append((c, U))
            t += 1
    b.philox(11, 0, 0)
    b.evolve(coupling, jw.SIN_KERNEL, 1e-4, nsteps=2, reunit_every=10)
    b.sync()
    for t, (c, U) in enumerate(singles):
        got = c.field()
        b.get(t, got)
        assert worst(got.download(), U.download()) <= 1e-13 * (2.0 ** 22 if mixed else 1.0), t
    b.close()
