"""Moves of the SVO traversal through the leaf grid (pops and descents by
cell coordinates) against the oracle's node walk, bit for bit, step counts
included: origins on cell, node and root boundaries, outside the root and not
finite; directions along axes, with equal components, zero, denormal, tiny
and huge ones; the smallest and largest tree depths."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
import tg_amd as T
from tests import scenes as S
from tests.test_gpu_svo import assert_same_hits

pytestmark = pytest.mark.gpu

F = np.float32


def edge_rays(rng, mn, side, n, box):
    """n rays about [box[0], box[1]]^3 of the root [mn, mn + side)^3: origins
    on multiples of 32 and up to 3 ulps beside them, on the root's faces and
    corners, and outside."""
    o = rng.uniform(box[0], box[1], (n, 3))
    k = np.arange(n)
    o = np.where((rng.random((n, 3)) < 0.5) & (k % 3 == 0)[:, None], mn + 32.0 * np.round((o - mn) / 32.0), o)
    o[k % 7 == 1] = np.clip(mn + side * rng.integers(0, 3, (n, 3))[k % 7 == 1] / 2.0, mn - 1, mn + side + 1)
    o[k % 11 == 2] += rng.choice((-1.0, 1.0), (int((k % 11 == 2).sum()), 3)) * side
    o = o.astype(F)
    for _ in range(3):
        m = rng.random((n, 3)) < 0.2
        o = np.where(m, np.nextafter(o, np.where(rng.random((n, 3)) < 0.5, F(-1e9), F(1e9))), o)
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    sgn = np.where(rng.random((n, 3)) < 0.5, -1.0, 1.0)
    d[k % 5 == 0] = sgn[k % 5 == 0] * np.abs(d[k % 5 == 0, :1])
    d[k % 5 == 1] *= rng.choice((0.0, 1.0), (int((k % 5 == 1).sum()), 3))
    d[k % 5 == 2] *= rng.choice((1.0, 1e-7, 1e-31, 1e-39), (int((k % 5 == 2).sum()), 3))
    d[k % 5 == 3] *= rng.choice((1.0, 1e8, 1e15, 1e-20), (int((k % 5 == 3).sum()), 1))
    return o, d.astype(F)


@pytest.mark.parametrize("depth", [6, 9, 13])
def test_moves_equal_oracle(ctx, depth):
    rng = np.random.default_rng(100 + depth)
    side = float(1 << depth)
    mn = np.floor(np.array([-0.37, 0.11, -0.5]) * side)
    centres = mn + side * np.array([[0.5, 0.5, 0.5], [0.52, 0.45, 0.55], [0.5, 0.6, 0.5]])
    sc = S.make_scene([{"n": (2, 3, 2), "translation": tuple(c), "rotation": S.random_rotation(rng)} for c in centres],
                      seed=depth)
    ctx.upload(sc)
    ctx.svo_build(mn, depth)
    ref = O.OracleSvo(O.OracleScene(sc), mn.astype(F), depth)
    o, d = edge_rays(rng, mn, side, 12000, (mn.min() + 0.3 * side, mn.max() + 0.8 * side))
    o[:64] = np.where(rng.random((64, 3)) < 0.2, rng.choice((1e30, -1e30), (64, 3)), o[:64])
    wild_o, wild_d = o[:256].copy(), d[:256].copy()
    wild_o[:128] = np.where(rng.random((128, 3)) < 0.3, rng.choice((np.nan, np.inf, -np.inf), (128, 3)), wild_o[:128])
    wild_d[128:] = np.where(rng.random((128, 3)) < 0.3, rng.choice((np.nan, np.inf, -np.inf), (128, 3)), wild_d[128:])
    old = ctx.tuning()
    wild = []
    try:
        for dda in (0, 1):
            ctx.set_tuning(trace_dda=dda)
            for reach in (3.0e38, 0.3 * side):
                print(f"depth {depth} dda {dda} reach {reach}", flush=True)
                with np.errstate(all="ignore"):
                    want = ref.trace(o, d, reach)
                assert_same_hits(ctx.svo_trace(o, d, reach), want, f"depth {depth} dda {dda} reach {reach}")
            # inputs that are not finite: both forms of the leaf DDA agree (and end)
            wild.append(ctx.svo_trace(wild_o, wild_d, 3.0e38).tobytes())
    finally:
        ctx.set_tuning(trace_dda=int(old["trace_dda"][0]))
    assert wild[0] == wild[1]
    assert 30 <= want["hit"].sum() < 0.9 * len(o) and (np.abs(d).max(1) == 0.0).any()
