"""Tile lists that outgrow their buffer while a frame graph holds the
context's buffers: the call that overflows and every call after it still run
(an overflowing frame is exact, and its buffer grows only when it may)."""
from __future__ import annotations

import sys

import numpy as np
import pytest

import oracle as O
import tg_amd as T

pytestmark = pytest.mark.gpu

CAPACITY = 1 << 22          # entries of a first call's buffer
W, H, N = 960, 540, 64      # at 8x8 tiles more entries than that
w, h = 96, 64


def prepared(scene, corner):
    ctx = T.Context(0)
    ctx.upload(scene)
    ctx.svo_build(corner, 10)
    ctx.set_tuning(vis_tile=8)
    return ctx


def test_calls_after_an_overflow_under_a_frame_graph():
    p = T.noise_objects_params(seed=3, n_objects=512, max_extent=8, world=512.0)
    sc = T.generate_scene(p)
    cam = T.generate_camera(p, 0, w, h)
    corner = np.floor(cam[0]["camera"][:3]) - 512.0
    ref = O.visibility_brute(O.OracleScene(sc), cam, w, h)
    many = np.concatenate([T.generate_camera(p, i, W, H) for i in range(N)])
    full, got, words = np.empty((N, H, W), np.uint64), np.empty((N, H, W), np.uint64), np.empty((h, w), np.uint64)
    with prepared(sc, corner) as ctx:
        big = ctx.alloc(full.nbytes)
        for _ in range(2):                          # the second call's lists are whole
            ctx.visibility_device(many, W, H, big)
            assert ctx.last_stats().tile_entries > CAPACITY
        ctx.d2h(full, big)
        ctx.free(big)
    with prepared(sc, corner) as ctx:
        big, small = ctx.alloc(full.nbytes), ctx.alloc(8 * w * h)
        rad, irr = ctx.alloc(12 * w * h), ctx.alloc(12 * w * h)

        def check_small(what):
            print(f"[gpu] {what}", file=sys.stderr, flush=True)
            ctx.visibility_device(cam, w, h, small)
            ctx.d2h(words, small)
            assert np.array_equal(words, ref), what

        def check_big(what):
            print(f"[gpu] {what}", file=sys.stderr, flush=True)
            ctx.visibility_device(many, W, H, big)
            ctx.d2h(got, big)
            assert np.array_equal(got, full), what

        ctx.set_list_capacity(CAPACITY)
        check_big("every buffer but the lists' is large enough")
        gi = T.gi_params(T.seeded_sun(3), spp=1, max_distance=512.0)
        with ctx.frame_graph(cam, w, h, gi, small, rad, irr) as graph:
            ctx.set_list_capacity(0)
            check_small("before the overflow")
            for i in range(2):
                check_big(f"overflow {i}")
                for k in range(2):
                    check_small(f"call {k} after it")
            graph.launch()
            ctx.d2h(words, small)
            assert np.array_equal(words, ref)
        check_small("without the graph the buffer may grow again")
        check_big("in full")
        for q in (big, small, rad, irr):
            ctx.free(q)
