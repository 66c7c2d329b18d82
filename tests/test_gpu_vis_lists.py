"""Tile lists of visibility about the lengths where their sorting and staging
change (64 records a stage, 128 keys sorted by rank, 1024 a chunk): clusters in
one tile, front to back and behind one another, against the oracle, word for
word."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from tests import scenes as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 127, 128, 129, 257, 1025])
def test_list_lengths(ctx, n):
    rng = np.random.default_rng(n)
    objs = [{"n": (1, 1, 1), "translation": tuple(np.array([0.0, 0.0, 0.0]) + rng.uniform(-20, 20, 3)),
             "rotation": S.random_rotation(rng)} for _ in range(n)]
    bits = [np.packbits(rng.random(512) < 0.02, bitorder="little").view(np.uint32) for _ in range(n)]
    for b in bits:
        b[0] |= np.uint32(1)
    sc = S.make_scene(objs, bits_per_cluster=bits, seed=n)
    ctx.upload(sc)
    cam = S.axis_camera((0.0, 0.0, 90.0), 2, -1.0)
    print(f"{n} clusters", flush=True)
    want = O.visibility_brute(O.OracleScene(sc), cam, 32, 32)
    assert np.array_equal(ctx.visibility(cam, 32, 32)[0], want)
    assert (want != np.uint64(0xFFFFFFFFFFFFFFFF)).any()
