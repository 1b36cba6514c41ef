"""The large lattices in every coupling and noise space, on the column strips that run by
default against the 16-byte ones, and the matrix-core stages where they are asked for."""
import numpy as np
import pytest

from test_gpu_colreg import CORR, FIXED, NOISE, SQRT, bound, evolved, start, worst

pytestmark = pytest.mark.gpu

NARROW = 8      # fused mode: one plane at a time over 16-byte strips
ROW_MAJOR = 2


# two steps: the first leaves U in the storage type, the last the whole FP64 field
@pytest.mark.parametrize("space,coupling", [("position", SQRT), ("position", NOISE), ("position", FIXED), ("position", CORR),
                                            ("momentum", SQRT), ("momentum", FIXED), ("momentum", CORR)])
@pytest.mark.parametrize("N,mixed", [(4096, 0), (4096, 1), (8192, 1)])
def test_default_strips_match_narrow_ones(jw, N, mixed, space, coupling):
    c, U0 = start(jw, N)
    noise = jw.NOISE_MOMENTUM if space == "momentum" else jw.NOISE_POSITION
    a = evolved(jw, c, U0, jw.Context.FUSED, noise, coupling, mixed)
    b = evolved(jw, c, U0, NARROW, noise, coupling, mixed)
    c.close()
    assert worst(a, b) <= bound(N, mixed)


# split BF16: about 2^-17 a stage (the bound of the mixed form's S(r)); FP32 butterflies 3e-7
@pytest.mark.parametrize("space", ["position", "momentum"])
def test_matrix_core_stages_run_on_row_major_planes(jw, space):
    c, U0 = start(jw, 4096)
    noise = jw.NOISE_MOMENTUM if space == "momentum" else jw.NOISE_POSITION
    exact = evolved(jw, c, U0, jw.Context.FUSED, noise, CORR, 0)
    c.set_mixed_fft(1)
    err = [worst(evolved(jw, c, U0, mode, noise, CORR, 1), exact) for mode in (ROW_MAJOR, NARROW)]
    c.close()
    assert all(1e-6 < e < 2e-5 for e in err), err
