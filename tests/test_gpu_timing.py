"""Kernel timing around calls that run several host threads."""
import pytest

pytestmark = pytest.mark.gpu


# N = 64: one lane; 512 and 1024: the symmetrised reals pass through four lanes, a host thread each
@pytest.mark.parametrize("N", [64, 512, 1024])
def test_a_measurement_is_one_timed_call(jw, N):
    c = jw.Context(N)
    U = c.field()
    c.set_unit(U)
    c.timing(True)
    for k in range(1, 6):
        c.measure_corr(U)
        # the correlator's passes are timed once, on the calling thread; no lane adds to the counters
        assert c.kernel_times()["observables"][1] == k
    c.close()
