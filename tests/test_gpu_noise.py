"""The normals of the Philox stream on the GPU against an extended-precision
Box-Muller on the same words."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

L = np.longdouble


def philox(c, k0, k1):
    """Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11) on uint64 arrays of 32-bit words."""
    m = np.uint64(0xFFFFFFFF)
    for r in range(10):
        p0 = np.uint64(0xD2511F53) * c[0]
        p1 = np.uint64(0xCD9E8D57) * c[2]
        a, b = np.uint64((k0 + r * 0x9E3779B9) & 0xFFFFFFFF), np.uint64((k1 + r * 0xBB67AE85) & 0xFFFFFFFF)
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ a, p1 & m, (p0 >> np.uint64(32)) ^ c[3] ^ b, p0 & m]
    return c


@pytest.mark.parametrize("N,seed,traj,step", [(64, 1, 0, 0), (512, 0xFFFFFFFF, 7, 3), (1024, 12345, 0x80000000, 99)])
def test_normals_match_extended_precision(jw, N, seed, traj, step):
    ctx = jw.Context(N)
    ctx.philox(seed, traj, step)
    xx, xy = ctx.field(), ctx.field()
    ctx.generate_gaussian(xx, xy)
    site = np.arange(N * N, dtype=np.uint64)
    # call 0 gives n0, m0: the real part of entry 1 of xi_x and xi_y
    c = philox([site, np.full_like(site, step), np.full_like(site, jw.TAG_LANGEVIN), np.zeros_like(site)], seed, traj)
    a = ((c[0] << np.uint64(32)) | c[1]) >> np.uint64(11)
    b = ((c[2] << np.uint64(32)) | c[3]) >> np.uint64(11)
    # u0 is rounded to FP64 once before its logarithm; the angle is exact
    u0 = ((a.astype(L) + L(0.5)) * L(2) ** -53).astype(np.float64).astype(L)
    r = np.sqrt(-2 * np.log(u0))
    turn = 2 * np.arctan2(L(0), L(-1)) * (b.astype(L) + L(0.5)) * L(2) ** -53
    for got, ref in ((xx, r * np.cos(turn)), (xy, r * np.sin(turn))):
        z = got.download()[:, 1].real.astype(L)
        # logarithm 1 ulp (half of it in the radius), square root, sine or cosine and product 1, 1
        # and 1/2 ulp: 3 units of 2^-53 relative to r, doubled for slack
        assert (np.abs(z - ref) <= 6 * L(2) ** -53 * np.maximum(r, L(2) ** -26)).all()
    ctx.close()


def test_normals_are_white(jw):
    """The sixteen normals of a site: unit variance, no correlation (5 sigma of the sample size)."""
    N = 512
    ctx = jw.Context(N)
    ctx.philox(5, 1, 2)
    xx, xy = ctx.field(), ctx.field()
    ctx.generate_gaussian(xx, xy)
    z = []
    for f in (xx, xy):
        u = f.download()
        z += [u[:, 1].real, u[:, 1].imag, (u[:, 0].real - u[:, 4].real) / 2, u[:, 2].real, u[:, 2].imag, u[:, 5].real,
              u[:, 5].imag, -u[:, 8].real * np.sqrt(3.0) / 2]
    C = np.cov(np.array(z))
    assert np.abs(C - np.eye(16)).max() <= 5 * np.sqrt(2.0 / (N * N))
    ctx.close()
