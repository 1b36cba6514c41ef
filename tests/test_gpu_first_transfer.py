"""The first transfers of a fresh context: exact, and without the price of the pinned
buffers that later ones use."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# N = 128: three chunks through the device buffer; 256 (nine components): pinned lanes at once
@pytest.mark.parametrize("t", [1, 9])
@pytest.mark.parametrize("N", [4, 16, 64, 128, 256])
def test_each_first_call_is_exact(jw, N, t):
    a = np.random.default_rng(N + t).normal(size=(N * N, t, 2)).view(np.complex128)[..., 0]
    c = jw.Context(N)
    f = c.field(t)
    for k in range(6):                       # the device buffer, then the lanes
        f.upload(a + k)
        assert np.array_equal(f.download(), a + k)
    c.close()
    if t == 9:                               # a download, a measurement first
        c = jw.Context(N)
        f = c.field()
        c.set_unit(f)
        assert np.array_equal(f.download(), np.tile(np.eye(3).reshape(9), (N * N, 1)))
        c.close()
        c = jw.Context(N)
        f = c.field()
        c.set_unit(f)
        first = c.measure_corr(f)
        assert first[0] > 0 and all(np.array_equal(first, c.measure_corr(f)) for _ in range(5))
        c.close()


def test_a_first_upload_costs_no_pinned_allocation(jw):
    N = 64
    a = np.ones((N * N, 9), np.complex128)
    first, later = [], []
    for _ in range(21):
        c = jw.Context(N)
        f = c.field()
        c.sync()
        for times in [first] + 8 * [[]] + [later]:
            t0 = time.perf_counter()
            f.upload(a)
            times.append(time.perf_counter() - t0)
        c.close()
    # one pinned buffer takes 32 us; four of them and their events took 96 us here
    assert np.median(first) - np.median(later) <= 30e-6
