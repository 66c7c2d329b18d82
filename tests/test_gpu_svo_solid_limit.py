"""SVOs of nearly and of more than 2^32 solid voxels, the range of the leaves'
material offsets: the one equals the builds of its octants, in counts and in the
bounce light of the last octant, whose materials come last; the other is
refused, and the context builds on."""
from __future__ import annotations

import sys

import numpy as np
import pytest

import tg_amd as T

pytestmark = pytest.mark.gpu

SIDE, SCALE = 8192.0, 16.0


def scene(n):
    """n clusters of 16^3 world voxels a voxel, half of them solid, rotated about z."""
    rng = np.random.default_rng(6)
    a = rng.uniform(0.0, 2.0 * np.pi, n)
    objects = np.zeros(n, T.OBJECT_DTYPE)
    objects["n_cluster_pointers_per_dim"] = 1
    objects["first_cluster_pointer"] = np.arange(n)
    objects["translation"] = rng.uniform(100.0, SIDE - 100.0, (n, 3))
    rot = np.zeros((n, 4, 4), np.float32)
    rot[:, 0, 0] = rot[:, 1, 1] = SCALE * np.cos(a)
    rot[:, 0, 1], rot[:, 1, 0] = SCALE * np.sin(a), -SCALE * np.sin(a)
    rot[:, 2, 2], rot[:, 3, 3] = SCALE, 1.0
    objects["rotation"] = rot.reshape(n, 16)
    bits = np.packbits(rng.random((n, 512)) < 0.5, axis=1, bitorder="little").view(np.uint32)
    luts = np.zeros(256, T.LUT_DTYPE)
    luts["albedo"] = rng.uniform(0.1, 0.9, (256, 3))
    idx = np.arange(n, dtype=np.uint32)
    sc = T.Scene(objects, idx, idx.copy(), bits.ravel(), rng.integers(0, 256, 512 * n, dtype=np.uint8), luts)
    return sc, int(np.unpackbits(bits.view(np.uint8)).sum()) * 4096


def totals(ctx):
    info = ctx.svo_info()
    return np.array([info["n_leaves"], info["n_list_entries"], ctx.svo_device_bytes()[1]], np.int64)


def test_below_the_limit():
    sc, voxels = scene(4000)                  # overlapping voxels count once
    assert 0.96 * 2 ** 32 < voxels < 2 ** 32
    w, h = 480, 270
    with T.Context(0) as ctx:
        ctx.upload(sc)
        cam = T.make_camera((6144.0, 6144.0, 6144.0), 0.3, 0.7, 0.0, 1.2, w / h, 0.1, 1900.0)
        gi = T.gi_params(T.seeded_sun(5), spp=8, max_distance=1900.0)
        parts = np.zeros(3, np.int64)
        for o in range(8):
            print(f"[gpu] octant {o}", file=sys.stderr, flush=True)
            ctx.svo_build([SIDE / 2 * ((o >> a) & 1) for a in range(3)], 12)
            parts += totals(ctx)
        vis, rad, irr = ctx.frame(cam, w, h, gi)
        print(f"[gpu] whole root, {parts}", file=sys.stderr, flush=True)
        assert 0.9 * 2 ** 32 < parts[2] <= voxels
        ctx.svo_build((0.0, 0.0, 0.0), 13)
        assert np.array_equal(totals(ctx), parts)
        vis2, rad2, irr2 = ctx.frame(cam, w, h, gi)
    assert np.array_equal(vis, vis2)
    lit = irr.any(-1) | irr2.any(-1)
    same = (rad == rad2).all(-1) & (irr == irr2).all(-1)
    print(f"[gpu] lit {lit.sum()}, same {same[lit].mean()}", file=sys.stderr, flush=True)
    # positions are held relative to the root's centre: a ray may round to another voxel
    assert lit.sum() > 1000 and same[lit].mean() > 0.9


def test_beyond_the_limit():
    sc, voxels = scene(4700)
    assert voxels > 1.12 * 2 ** 32            # more than overlaps take off
    with T.Context(0) as ctx:
        ctx.upload(sc)
        print("[gpu] whole root", file=sys.stderr, flush=True)
        with pytest.raises(T.TgxError, match="solid voxels"):
            ctx.svo_build((0.0, 0.0, 0.0), 13)
        with pytest.raises(T.TgxError):
            ctx.svo_info()
        print("[gpu] an octant", file=sys.stderr, flush=True)
        ctx.svo_build((0.0, 0.0, 0.0), 12)
        assert totals(ctx)[2] > 0
