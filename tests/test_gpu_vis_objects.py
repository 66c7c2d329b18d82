"""Visibility on both sides of the object count from which the objects are
culled by a grid of their own instead of one workgroup per camera: several
cameras, so that each camera's block of the object lists counts, through the
ordinary, the host-array and the allocation-free entry points; words equal the
oracle's."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
import tg_amd as T
from tests import scenes as S

pytestmark = pytest.mark.gpu

W, H, CAMS = 160, 90, 3


@pytest.mark.parametrize("n", [3071, 3072, 3073, 4097, 5000])
def test_object_cull_forms(ctx, n):
    rng = np.random.default_rng(n)
    at = rng.uniform(-160.0, 160.0, (n, 3))
    at[-1] = (0.0, 0.0, -30.0)           # the last object is in view
    sc = S.make_scene([{"n": (1, 1, 1), "translation": tuple(p), "rotation": S.random_rotation(rng)} for p in at], seed=n)
    sc.bits[: 16 * 40] = 0               # objects without a solid voxel are none of the kept ones
    ctx.upload(sc)
    # the first camera looks at the last object, from outside most of the others
    cams = np.concatenate([T.make_camera((0.0, 0.0, 0.0), 0.0, a, 0.0, 1.2, W / H, 0.1, 400.0) for a in (0.0, 2.1, 4.2)])
    os_ = O.OracleScene(sc)
    want = np.stack([O.visibility_culled(os_, cams[i:i + 1], W, H)[0] for i in range(CAMS)])
    assert 0.02 < (want != T.VISIBILITY_EMPTY).mean() < 0.98
    print(f"[gpu] {n} objects, {CAMS} cameras {W}x{H}", flush=True)
    assert np.array_equal(ctx.visibility(cams, W, H), want)
    assert np.array_equal(ctx.visibility(cams[1:2], W, H)[0], want[1])
    dev = ctx.alloc(want.nbytes)
    try:
        ctx.visibility_device_noalloc(cams, W, H, dev)
        got = np.empty_like(want)
        ctx.d2h(got, dev)
        assert np.array_equal(got, want)
    finally:
        ctx.free(dev)
    last = (want >> np.uint64(9)) & np.uint64(0x7FFFFFFF)
    assert ((last == n - 1) & (want != T.VISIBILITY_EMPTY)).any()
