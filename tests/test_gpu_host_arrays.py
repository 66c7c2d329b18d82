"""Calls on host arrays pass them through pinned memory that the kernels read,
256 records a block, in pieces of 4 MiB: odd counts about a block's edge, a call
after a larger one, and one of many pieces, whose results are those of the same
records in small calls, bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
import tg_amd as T
from tests import scenes as S
from tests.test_gpu_svo import assert_same_hits, rays_from

pytestmark = pytest.mark.gpu


def test_trace_counts(ctx):
    rng = np.random.default_rng(4)
    sc = S.make_scene([{"n": (3, 2, 3), "translation": tuple(rng.uniform(10, 118, 3)), "rotation": S.random_rotation(rng)}
                       for _ in range(9)], seed=4)
    ctx.upload(sc)
    ctx.svo_build((0.0, 0.0, 0.0), 7, 0)
    ref = O.OracleSvo(O.OracleScene(sc), (0.0, 0.0, 0.0), 7, 0)
    for n in (1, 255, 256, 257, 3001, 64):
        print(f"{n} rays", flush=True)
        o, d = rays_from(rng, max(n, 8), -10, 140, centre=(64.0, 64.0, 64.0))
        assert_same_hits(ctx.svo_trace(o[:n], d[:n], 300.0), ref.trace(o[:n], d[:n], 300.0), f"{n} rays")
    n = 600_001
    print(f"{n} rays", flush=True)
    o, d = rays_from(rng, n, -10, 140)
    big = ctx.svo_trace(o, d, 300.0)
    for a in (0, 299_999, n - 1000):
        assert_same_hits(big[a:a + 1000], ctx.svo_trace(o[a:a + 1000], d[a:a + 1000], 300.0), "in many pieces")


def test_cache_counts(ctx):
    rng = np.random.default_rng(5)
    s = rng.uniform(-1, 1, (800_001, 9)).astype(np.float32)
    s[:, 3:6] /= np.linalg.norm(s[:, 3:6], axis=1, keepdims=True)
    s[:, 6:] = np.abs(s[:, 6:])

    def infer(a, n):
        return ctx.nrc_infer(s[a:a + n, :3], s[a:a + n, 3:6], s[a:a + n, 6:]).view(np.uint32)

    def step(n):
        ctx.nrc_create(T.nrc_config())
        loss, grad = ctx.nrc_train_batch(s[:n, :3], s[:n, 3:6], s[:n, 6:], np.abs(s[:n, :3]), want_grad=True)
        assert np.isfinite(loss) and np.isfinite(grad).all() and grad.any()
        return loss, grad, ctx.nrc_params()

    counts = (1, 255, 256, 257)
    ctx.nrc_create(T.nrc_config())
    first = infer(0, 1)
    before = [step(n) for n in counts]
    ctx.nrc_create(T.nrc_config())
    print("inference in many pieces", flush=True)
    big = infer(0, len(s))
    assert np.array_equal(big[:1], first)
    for a, n in ((16, 255), (0, 256), (777, 257), (797_000, 3001)):
        print(f"inference of {n}", flush=True)
        assert np.array_equal(infer(a, n), big[a:a + n]), n
    for n, ref in zip(counts, before):
        print(f"a step on {n}", flush=True)
        for x, y in zip(step(n), ref):
            assert np.array_equal(x, y)
