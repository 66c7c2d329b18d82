"""Levels of the SVO build where their arrays and bitmaps can go wrong: the
smallest and the largest depth, a level with more (node, cluster) pairs than
the arrays hold at first, a scene after such a one, no solid cluster at all,
and more leaves than one block scans; against the oracle's build, byte for
byte, where it is small enough to run."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
import tg_amd as T
from tests import scenes as S
from tests.test_gpu_svo import assert_same_svo

pytestmark = pytest.mark.gpu


def scaled(rng, n, extent, scale, at):
    objs = []
    for _ in range(n):
        r = np.asarray(S.random_rotation(rng), np.float32).reshape(4, 4).copy()
        r[:3, :3] *= scale
        objs.append({"n": extent, "translation": tuple(at + rng.uniform(-6, 6, 3)), "rotation": r.reshape(16)})
    return objs


def same(ctx, sc, mn, depth):
    ctx.svo_build(mn, depth, 0)
    assert_same_svo(ctx.svo_export(), O.OracleSvo(O.OracleScene(sc), mn, depth, 0).export(), f"depth {depth}")


@pytest.mark.parametrize("depth, at", [(6, 30.0), (7, 70.0), (9, 200.0), (11, 1900.0), (12, 4000.0), (13, 8100.0)])
def test_depths(ctx, depth, at):
    sc = S.make_scene(scaled(np.random.default_rng(depth), 5, (2, 1, 2), 1.0, at), seed=depth)
    ctx.upload(sc)
    print(f"depth {depth}", flush=True)
    same(ctx, sc, (0.0, 0.0, 0.0), depth)


def test_more_pairs_than_room(ctx):
    big = S.make_scene(scaled(np.random.default_rng(1), 40, (1, 1, 1), 20.0, 256.0), seed=1)
    small = S.make_scene(scaled(np.random.default_rng(2), 9, (2, 2, 2), 1.0, 256.0), seed=2)
    for what, sc in (("big", big), ("small", small), ("big again", big)):
        ctx.upload(sc)
        for k in range(2):
            print(f"{what}, build {k}", flush=True)
            same(ctx, sc, (0.0, 0.0, 0.0), 9)


def test_no_solid_cluster(ctx):
    sc = S.make_scene([{"n": (2, 2, 2), "translation": (30.0, 30.0, 30.0)}],
                      bits_per_cluster=[np.zeros(16, np.uint32)] * 8)
    ctx.upload(sc)
    same(ctx, sc, (0.0, 0.0, 0.0), 7)


def test_more_leaves_than_one_block_scans(ctx):
    sc = S.make_scene(scaled(np.random.default_rng(3), 1, (1, 1, 1), 130.0, 1024.0), seed=3)
    sc.materials[:] = 1 + np.arange(sc.materials.size).reshape(sc.materials.shape) % 5
    ctx.upload(sc)
    print("one cluster of 1040^3", flush=True)
    ctx.svo_build((0.0, 0.0, 0.0), 11, 0)
    e = ctx.svo_export()
    n = e["info"]["n_leaves"]
    assert n > 16384
    assert np.array_equal(e["list_offsets"][: n + 1], np.concatenate([[0], np.cumsum(e["leaf_n"])]))
    assert e["info"]["n_list_entries"] == int(e["leaf_n"].sum())
    pick = np.r_[0:n:997, n - 40:n]
    solid = np.unpackbits(np.ascontiguousarray(e["bits"][pick]).view(np.uint8), axis=1, bitorder="little")
    assert solid.any() and np.array_equal(np.asarray(e["materials"][pick]).reshape(len(pick), -1) != 0, solid != 0)
