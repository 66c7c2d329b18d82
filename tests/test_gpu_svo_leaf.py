"""Leaf sampling of the SVO build where its staging and its keys can go wrong:
leaves with more candidate clusters than one stage holds (64), with exactly a
stage, with several objects in the same place (the first candidate's material
wins), with scaled and mirrored objects and without materials; against the
oracle's build, byte for byte."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
import tg_amd as T
from tests import scenes as S
from tests.test_gpu_svo import assert_same_svo

pytestmark = pytest.mark.gpu


def overlapping(rng, n, extent, scale=1.0):
    """n objects about one point; their clusters share the leaves around it."""
    objs = []
    for _ in range(n):
        r = np.asarray(S.random_rotation(rng), np.float32).reshape(4, 4).copy()
        r[:3, :3] *= scale
        objs.append({"n": extent, "translation": tuple(16.0 + rng.uniform(-6, 6, 3)), "rotation": r.reshape(16)})
    return objs


@pytest.mark.parametrize("n, extent, scale", [(1, (4, 4, 4), 1.0), (8, (2, 2, 2), 1.0), (9, (2, 2, 2), 1.0),
                                              (40, (2, 3, 1), 1.0), (6, (2, 2, 2), -1.0), (5, (3, 3, 3), 0.3),
                                              (3, (1, 1, 1), 4.0)])
@pytest.mark.parametrize("materials", [True, False])
def test_leaf_sampling_equals_oracle(ctx, n, extent, scale, materials):
    rng = np.random.default_rng(n)
    sc = S.make_scene(overlapping(rng, n, extent, scale), seed=n)
    if materials:
        ctx.upload(sc)
    else:
        d = sc.desc()
        d.materials = None
        ctx._check(ctx.lib.tgx_scene_upload(ctx.h, d), "tgx_scene_upload")
        sc.materials[:] = 0
    mn = (-48.0, -48.0, -48.0)
    for quirk in (0, T.SVO_FLAG_REFERENCE_CORNER_QUIRK):
        print(f"{n} objects of {extent}, scale {scale}, materials {materials}, quirk {quirk}", flush=True)
        ctx.svo_build(mn, 7, quirk)
        assert_same_svo(ctx.svo_export(), O.OracleSvo(O.OracleScene(sc), mn, 7, quirk).export(), "overlap")
