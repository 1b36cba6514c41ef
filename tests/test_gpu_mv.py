"""The MV start (jw_mv_init) at every size of its fused passes and beside them, against
the same sheets through the per-function calls."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("injected", [0, 1])
@pytest.mark.parametrize("N,sheets,zero", [(32, 2, 0), (64, 1, 1), (64, 3, 0), (128, 2, 0), (256, 3, 1), (512, 2, 0),
                                           (1024, 1, 1), (2048, 2, 0), (4096, 1, 1)])
def test_sheets_match_per_function_calls(jw, N, sheets, zero, injected):
    """A mass above the lattice's largest momentum (m = 4, phat^2 <= 8): no mode is near the
    pole of the Poisson factor, which lies in [1/16, 1/8], so the potential is at most
    sigma / 8 times a normal and the exponential needs no squaring."""
    g, mu, mass = 1.0, 4.0, 1.0
    c = jw.Context(N)
    c.set_mv_zero_mode(zero)
    z = np.random.default_rng(N + sheets).normal(size=(sheets, N * N * 8)) if injected else None
    U = c.field()
    c.philox(5, 2, 0)
    c.mv_init(U, sheets, g, mu, mass, z)
    V, f = c.field(), c.field()
    c.set_unit(V)
    c.philox(5, 2, 0)
    for s in range(sheets):
        if injected:
            c.inject(z[s], 8)
        c.set_mv_model(f, g, mu, sheets)
        c.execute2D(f, 1)
        c.solve_poisson(f, mass * g * g * mu, g)
        c.execute2D(f, 0)
        c.mul_exp(V, f)
    a, b = U.download(), V.download()
    # per site and sheet: a potential of norm below 10 with the rounding of two transforms on
    # either side (4 log2(N^2) 2^-53 of it), an exponential and a product (40 2^-53)
    bound = sheets * (10 * 4 * np.log2(N * N) + 2 * 40) * 2.0 ** -53
    assert np.sqrt((np.abs(a - b) ** 2).sum(axis=1)).max() <= bound
    u = a.reshape(-1, 3, 3)
    assert np.abs(u @ u.conj().transpose(0, 2, 1) - np.eye(3)).max() < 1e-14 * (1 + sheets)
    assert np.abs(a - np.eye(3).reshape(9)).max() > 0.1
    c.close()
