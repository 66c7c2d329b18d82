"""The uncounted leaf walk takes its voxels several at a time: leaves so full
or so empty that it ends at each place of such a group, by a hit, by an exit or
after crossing bricks, with bursts of fewer voxels than a group, of one and of
several, against the oracle's walk bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from tests import scenes as S
from tests.test_gpu_svo import assert_same_hits, rays_from

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fill", [0.5, 0.06, 0.004])
def test_groups_of_voxels(ctx, fill):
    rng = np.random.default_rng(int(1000 * fill))
    objs = [{"n": (4, 4, 4), "translation": tuple(c), "rotation": S.random_rotation(rng)}
            for c in ((40.0, 40.0, 40.0), (80.0, 60.0, 70.0), (60.0, 90.0, 50.0))]
    bits = [np.packbits(rng.random(512) < fill, bitorder="little").view(np.uint32) for _ in range(3 * 64)]
    sc = S.make_scene(objs, bits_per_cluster=bits, seed=1)
    ctx.upload(sc)
    ctx.svo_build((0.0, 0.0, 0.0), 7, 0)
    ref = O.OracleSvo(O.OracleScene(sc), (0.0, 0.0, 0.0), 7, 0)
    o, d = rays_from(rng, 6000, 20, 110, centre=(60.0, 60.0, 60.0))
    want = ref.trace(o, d, 300.0)
    old = ctx.tuning()
    try:
        for burst in (2, 6, 8, 18, 32):
            for cross in (0, 1, 64):
                print(f"fill {fill} burst {burst} cross {cross}", flush=True)
                ctx.set_tuning(trace_dda=1, trace_burst=burst, trace_cross=cross)
                assert_same_hits(ctx.svo_trace(o, d, 300.0), want, f"burst {burst} cross {cross}")
    finally:
        ctx.set_tuning(**{k: int(old[k][0]) for k in old.dtype.names})
