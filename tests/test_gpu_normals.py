"""The normals of both noise streams in both precisions, from given Philox words, against
an extended-precision Box-Muller: random words, and uniforms next to 0, 1/2 and 1 with
angles next to every eighth of a turn."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

L = np.longdouble


def words():
    w = np.random.default_rng(1).integers(0, 1 << 32, (200_000, 4), dtype=np.uint64)
    # 64-bit pairs at the edges: the upper 53 bits make the uniform
    top = [0, 1, 2, 1 << 20, (1 << 52) - 1, 1 << 52, (1 << 52) + 1, (1 << 53) - 1, (1 << 53) - 2, (1 << 53) - (1 << 29),
           (1 << 53) - (1 << 30), (1 << 53) - (1 << 21)]
    top += [k << 50 for k in range(1, 8)] + [(k << 50) - 1 for k in range(1, 8)]
    pairs = [((m << 11) >> 32, (m << 11) & 0xFFFFFFFF) for m in top]
    # 32-bit uniforms take each word by itself
    pairs += [(a, b) for a in (0, 1, 0x7FFFFFFF, 0x80000000, 0xFFFFFFFE, 0xFFFFFFFF) for b in (0, 0xFFFFFFFF)]
    edge = np.array([p + q for p in pairs for q in pairs], np.uint64)
    return np.concatenate([w, edge])


def exact(u0, u1):
    r, t = np.sqrt(-2 * np.log(u0)), 2 * np.arctan2(L(0), L(-1)) * u1
    return r, np.stack([r * np.cos(t), r * np.sin(t)], 1)


def test_normals_of_given_words(jw):
    w = words()
    c = jw.Context(64)
    got = c.box_muller(w).astype(L)
    c.close()
    m = [((w[:, 2 * k] << np.uint64(32)) | w[:, 2 * k + 1]) >> np.uint64(11) for k in (0, 1)]
    u = [(x.astype(L) + L(0.5)) * L(2) ** -53 for x in m]
    v = [(w[:, k].astype(L) + L(0.5)) * L(2) ** -32 for k in range(4)]
    # FP64: u0 is rounded once before its logarithm; then the logarithm 1 ulp (half of it in the
    # radius), square root, sine or cosine and product 1, 1 and 1/2: 3 units of 2^-53 relative to r, doubled
    r, z = exact(u[0].astype(np.float64).astype(L), u[1])
    assert (np.abs(got[:, 0:2] - z) <= 6 * L(2) ** -53 * np.maximum(r, L(2) ** -26)[:, None]).all()
    # FP32: the radius within 4 units of 2^-24 of max(r, 1), sine and cosine within 1.9e-7 (3.2
    # units) of the unit circle, the product half a unit: under 8 units of max(r, 1)
    r, z = exact(*u)
    assert (np.abs(got[:, 2:4] - z) <= 8 * L(2) ** -24 * np.maximum(r, 1)[:, None]).all()
    for p in (0, 1):
        r, z = exact(v[2 * p], v[2 * p + 1])
        assert (np.abs(got[:, 4 + 2 * p:6 + 2 * p] - z) <= 6 * L(2) ** -53 * r[:, None]).all()
        assert (np.abs(got[:, 8 + 2 * p:10 + 2 * p] - z) <= 8 * L(2) ** -24 * np.maximum(r, 1)[:, None]).all()
    # u0 next to 1: a radius of an FP32 ulp and less keeps its relative precision
    r, _ = exact(u[0], u[1])
    small = r < L(2) ** -13
    norm = np.sqrt((got[:, 2:4] ** 2).sum(axis=1))
    assert small.any() and (np.abs(norm - r)[small] <= 8 * L(2) ** -24 * r[small]).all()
