"""The phase vote (tuning trace_vote) over its whole range: a wave that runs
only moves or only leaf walks in a step still ends every ray, with the same
frame. Above 32 a wave may hold back its walking lanes for a few moving ones, so
a moving lane must never wait for others to move with it."""
from __future__ import annotations

import numpy as np
import pytest

import tg_amd as T

pytestmark = pytest.mark.gpu


def test_every_vote_gives_the_same_frame(ctx):
    p = T.noise_objects_params(seed=11, n_objects=40, max_extent=4, world=160.0)
    ctx.upload(T.generate_scene(p))
    cam = T.generate_camera(p, 0, 160, 90)
    ctx.svo_build(np.floor(cam[0]["camera"][:3]) - 256.0, 9)
    gi = T.gi_params(T.seeded_sun(11), spp=4, max_distance=400.0)
    want = ctx.frame(cam, 160, 90, gi)
    assert want[1].any()
    for dda in (1, 0):
        for vote in (1, 32, 33, 48, 63, 64):
            print(f"[gpu] vote {vote}, dda {dda}", flush=True)
            ctx.set_tuning(trace_vote=vote, trace_dda=dda)
            for a, b in zip(want, ctx.frame(cam, 160, 90, gi)):
                assert a.tobytes() == b.tobytes()
