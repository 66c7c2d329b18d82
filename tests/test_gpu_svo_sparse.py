"""SVO builds of many leaves with few candidate clusters each, where the
sampling passes change their form: leaves at the limits of candidates (15 to 17)
and of solid voxels (2048), in builds with fewer and with more than 1024
leaves and with fewer and more than 4 candidates a leaf; and updates of such
builds. Against the oracle's build, byte for byte."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
import tg_amd as T
from tests import scenes as S
from tests.test_gpu_svo import assert_same_svo

pytestmark = pytest.mark.gpu

MN = (0.0, 0.0, 0.0)
FULL = np.full(16, 0xFFFFFFFF, np.uint32)


def place(rng, n, lo, hi):
    """n random leaf cells of the 1024^3 root, their middles."""
    cells = rng.permutation(np.arange(lo, hi))[:n]
    return np.stack([cells % 32, cells // 32 % 32, cells // 1024], 1) * 32.0 + 16.0


def scene(rng, singles, knots):
    objs, bits = [], []

    def add(n, at, rotation, b=None):
        objs.append({"n": n, "translation": tuple(at), "rotation": rotation})
        for _ in range(int(np.prod(n))):
            bits.append(np.packbits(rng.random(512) < 0.3, bitorder="little").view(np.uint32) if b is None else b)

    for at in place(rng, singles, 0, 16384):
        add((1, 1, 1), at + rng.uniform(-12, 12, 3), S.random_rotation(rng))
    for at in place(rng, knots, 16384, 32768):
        for _ in range(int(rng.integers(15, 18))):                     # 15 to 17 candidates of one leaf
            add((1, 1, 1), at + rng.uniform(-1, 1, 3), S.random_rotation(rng))
    for at, n in zip(place(rng, 4, 16384, 32768), ((4, 1, 1), (2, 2, 1), (5, 1, 1), (2, 2, 2))):
        # whole clusters inside one leaf: 2048, 2048 and more solid voxels
        add(n, at if n[0] < 5 else at - (np.array(n) % 2) * 4.0, S.identity_rotation(), FULL)
    return S.make_scene(objs, bits_per_cluster=bits)


@pytest.mark.parametrize("singles, knots", [(300, 5), (1100, 20), (1100, 0), (500, 400)])
def test_sparse_builds_equal_the_oracle(ctx, singles, knots):
    sc = scene(np.random.default_rng(singles + knots), singles, knots)
    ctx.upload(sc)
    for quirk in (0, T.SVO_FLAG_REFERENCE_CORNER_QUIRK):
        print(f"{singles} clusters, {knots} knots, quirk {quirk}", flush=True)
        ctx.svo_build(MN, 10, quirk)
        got = ctx.svo_export()
        solid = np.unpackbits(np.ascontiguousarray(got["bits"]).view(np.uint8), axis=1).sum(1)
        assert (solid == 2048).any() and (solid > 2048).any()
        assert (got["info"]["n_leaves"] > 1024) == (singles + knots > 800)
        assert_same_svo(got, O.OracleSvo(O.OracleScene(sc), MN, 10, quirk).export(), "sparse")


def test_updates_of_a_sparse_build(ctx):
    rng = np.random.default_rng(9)
    sc = scene(rng, 1100, 20)
    n = len(sc.objects)
    ctx.scene_reserve(n + 4, sc.n_clusters + 64, sc.luts)
    live = []
    for o in sc.objects:
        f, k = int(o["first_cluster_pointer"]), int(np.prod(o["n_cluster_pointers_per_dim"]))
        live.append((ctx.object_create(o["n_cluster_pointers_per_dim"], o["translation"], o["rotation"], 0,
                                       sc.bits.reshape(-1, 16)[f:f + k], sc.materials.reshape(-1, 512)[f:f + k]), o, f, k))
    ctx.svo_build(MN, 10)
    for turn in range(3):
        idx, o, f, k = live[turn * 371]
        ctx.object_destroy(idx)
        o["translation"] += np.float32(3.0)
        ctx.object_create(o["n_cluster_pointers_per_dim"], o["translation"], o["rotation"], 0,
                          sc.bits.reshape(-1, 16)[f:f + k], sc.materials.reshape(-1, 512)[f:f + k])
        reused, sampled = ctx.svo_update()
        print(f"update {turn}: {reused} leaves kept, {sampled} sampled", flush=True)
        assert reused > 1024 and sampled > 0
        assert_same_svo(ctx.svo_export(), O.OracleSvo(O.OracleScene(ctx.scene_arrays()), MN, 10, 0).export(), f"update {turn}")
