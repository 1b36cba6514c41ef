"""Field upload and download through the pinned lanes: bit for bit, at sizes of one chunk
and of several, with a last chunk that is shorter, for both component counts."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# N = 64: one lane; 256: four lanes of one chunk; 512 and 1024: several chunks a lane,
# 4 MiB / 144 bytes does not divide the sites
@pytest.mark.parametrize("t", [1, 9])
@pytest.mark.parametrize("N", [4, 64, 128, 256, 512, 1024])
def test_round_trip_is_exact(jw, N, t):
    c = jw.Context(N)
    a = np.random.default_rng(N + t).normal(size=(2, N * N, t, 2)).view(np.complex128)[..., 0]
    f, g = c.field(t), c.field(t)
    for k in range(2):                    # the lanes' buffers are used again
        f.upload(a[k])
        assert np.array_equal(f.download(), a[k])
    c.copy(g, f)                          # device work before and after
    f.upload(a[0])
    assert np.array_equal(g.download(), a[1]) and np.array_equal(f.download(), a[0])
    if t == 9:                            # device planes hold what the per-site calls read
        c.set_unit(f)
        assert np.array_equal(f.download(), np.tile(np.eye(3).reshape(9), (N * N, 1)))
    c.close()
