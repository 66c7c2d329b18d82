"""An SVO of more leaves than one launch dimension takes at four workgroups of
512 lanes each: a root of 8192^3 voxels against the builds of its octants, whose
leaves are the same, and its bounce light against that of one octant."""
from __future__ import annotations

import sys

import numpy as np
import pytest

import tg_amd as T

pytestmark = pytest.mark.gpu


def totals(ctx):
    info = ctx.svo_info()
    return np.array([info["n_leaves"], info["n_list_entries"], ctx.svo_device_bytes()[1]], np.int64)


def test_leaves_beyond_two_million():
    p = T.noise_objects_params(seed=5, n_objects=1_800_000, max_extent=1, world=8100.0)
    w, h = 480, 270
    with T.Context(0) as ctx:
        ctx.generate_scene_device(p)
        # a camera in the middle of the last octant, whose leaves come last
        cam = T.make_camera((6144.0, 6144.0, 6144.0), 0.3, 0.7, 0.0, 1.2, w / h, 0.1, 1500.0)
        gi = T.gi_params(T.seeded_sun(5), spp=16, max_distance=1500.0)
        parts = np.zeros(3, np.int64)
        for o in range(8):
            corner = [4096.0 * ((o >> a) & 1) for a in range(3)]
            print(f"[gpu] octant {o}", file=sys.stderr, flush=True)
            ctx.svo_build(corner, 12)
            parts += totals(ctx)
        vis, rad, irr = ctx.frame(cam, w, h, gi)
        print(f"[gpu] whole root, {parts}", file=sys.stderr, flush=True)
        assert parts[0] > 1 << 21
        ctx.svo_build((0.0, 0.0, 0.0), 13)
        assert np.array_equal(totals(ctx), parts)
        vis2, rad2, irr2 = ctx.frame(cam, w, h, gi)
    assert np.array_equal(vis, vis2)
    lit = irr.any(-1) | irr2.any(-1)
    same = (rad == rad2).all(-1) & (irr == irr2).all(-1)
    print(f"[gpu] lit {lit.sum()}, same {same[lit].mean()}", file=sys.stderr, flush=True)
    # positions are held relative to the root's centre, so a ray in a hundred may
    # round to another voxel; a sample is its voxel's albedo and face, no position
    assert lit.sum() > 1000 and same[lit].mean() > 0.9
