"""The trace kernel skips the 32^3 leaf walk when a walk over the leaf's 8^3
bricks, in approximate crossing times, meets no brick holding a solid voxel
and every crossing is certain. This restates that test in float32 and holds it
to the exact walk (tg_amanatides_woo.c:3-114): a skipped leaf's walk never
enters such a brick. Entries on faces, edges and beside them; directions with
equal, nearly equal, tiny and zero components."""
import numpy as np
import pytest

F = np.float32


def entries(rng, n):
    d = rng.uniform(-1, 1, (n, 3))
    k = np.arange(n)
    d[k % 8 == 0] = rng.integers(-2, 3, ((k % 8 == 0).sum(), 3)) * 0.5
    d[k % 8 == 1, 1] *= 1e-6
    d[k % 8 == 2, 2] = 0.0
    m = k % 8 == 3
    d[m, 0] = d[m, 1] * (1 + rng.integers(-4, 5, m.sum()) * 2.0 ** -22)
    d[~d.any(1)] = (1.0, 0.0, 0.0)
    d = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(F)
    g = rng.uniform(0, 32, (n, 3))
    g = np.where((k % 4 == 1)[:, None], np.floor(g), np.where((k % 8 == 6)[:, None], np.floor(g) + 0.5, g))
    a = rng.integers(0, 3, n)
    g[k, a] = np.where(d[k, a] > 0, 0.0, 32.0) + rng.integers(-3, 4, n) * 1e-6 * rng.integers(0, 3, n)
    return g.astype(F), d


def leaf_clear(bm, g, d, v, td):
    b = v >> 3
    with np.errstate(over="ignore"):
        t = np.where(d > 0, (8 * b).astype(F) + F(8) - g, g - (8 * b).astype(F)) * td
    t = np.where(d == 0, F(3e38), t).astype(F)
    s = np.sort(t, 1)
    open_ = (t <= F(3e38)).all(1) & (s[:, 1] >= F(2.0 ** -100))
    clear = np.zeros(len(g), bool)
    sure = np.ones(len(g), F)
    step = np.where(d > 0, 1, -1)
    for _ in range(12):
        inside = ((b >= 0) & (b < 4)).all(1)
        clear |= open_ & ~inside & (sure > 0)
        open_ &= inside
        c = np.clip(b, 0, 3)
        open_ &= (bm >> (c[:, 0] + 4 * c[:, 1] + 16 * c[:, 2]).astype(np.uint64)) & np.uint64(1) == 0
        s = np.sort(t, 1)
        sure = np.minimum(sure, (s[:, 1].astype(np.float64) * (1 - 2.0 ** -17) - s[:, 0]).astype(F))
        ax = np.where(t[:, 0] == s[:, 0], 0, np.where(t[:, 1] == s[:, 0], 1, 2))
        k = np.arange(len(g))
        b[k, ax] += step[k, ax]
        t[k, ax] = (t[k, ax].astype(np.float64) + 8.0 * td[k, ax]).astype(F)
    return clear


def walk_touches(bm, g, d, v, td):
    v = v.copy()
    with np.errstate(divide="ignore", invalid="ignore", over="ignore"):
        tm = np.where(d > 0, (v + 1).astype(F) - g, g - v.astype(F)) / np.abs(d)
    tm = np.where(d == 0, F(3.402823466e38), tm).astype(F)
    step = np.sign(d).astype(int)
    live, touch = np.ones(len(g), bool), np.zeros(len(g), bool)
    k = np.arange(len(g))
    for _ in range(100):
        c = np.clip(v, 0, 31) >> 3
        touch |= live & ((bm >> (c[:, 0] + 4 * c[:, 1] + 16 * c[:, 2]).astype(np.uint64)) & np.uint64(1) != 0)
        x, y, z = tm.T
        ax = np.where(x < y, np.where(x < z, 0, 2), np.where(y < z, 1, 2))
        tm[k, ax] = np.where(live, tm[k, ax] + td[k, ax], tm[k, ax]).astype(F)
        v[k, ax] += np.where(live, step[k, ax], 0)
        live &= ((v >= 0) & (v < 32)).all(1)
    assert not live.any()
    return touch


@pytest.mark.parametrize("solid", [0.03, 0.2, 0.6])
def test_skipped_leaves_touch_no_solid_brick(solid):
    rng = np.random.default_rng(int(100 * solid))
    n = 60_000
    g, d = entries(rng, n)
    bits = rng.random((n, 64)) < solid
    bm = (bits.astype(np.uint64) << np.arange(64, dtype=np.uint64)).sum(1, dtype=np.uint64)
    v = np.clip(np.floor(g), 0, 31).astype(np.int64)
    with np.errstate(divide="ignore"):
        td = np.where(d == 0, F(3.402823466e38), F(1) / np.abs(d)).astype(F)
    clear, touch = leaf_clear(bm, g, d, v.copy(), td), walk_touches(bm, g, d, v, td)
    assert not (clear & touch).any()
    assert clear.sum() > 0.9 * (~touch).sum() > 0
