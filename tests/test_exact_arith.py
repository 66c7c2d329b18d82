"""Arithmetic that takes the place of IEEE divisions and of matrix products
and must give the same values: the quotient by a known reciprocal (every pair
of 24-bit significands whose quotient lies near the middle of two floats, where
alone it could round wrong, and random pairs), the floor of a division by a
host constant, and the cluster transforms of a rotation in a 4x4 matrix against
the products they leave out."""
import subprocess
from pathlib import Path

import numpy as np
import pytest

import tg_amd as T

CSRC = Path(T.__file__).resolve().parent / "csrc"

PROGRAM = r"""
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>
#include "tgx_m4.h"
#define __device__
struct dummy;
static uint32_t __float_as_uint(float f) { uint32_t u; memcpy(&u, &f, 4); return u; }
static uint32_t __umulhi(uint32_t a, uint32_t b) { return (uint32_t)(((uint64_t)a * b) >> 32); }
static uint32_t min(uint32_t a, uint32_t b) { return a < b ? a : b; }
static float __builtin_amdgcn_rcpf(float d) { return 1.0f / d; }
static float __builtin_amdgcn_rsqf(float d) { return 1.0f / sqrtf(d); }
#include "tgx_exact.h"

static uint64_t st = 88172645463325252ull;
static uint64_t rnd() { st ^= st << 13; st ^= st >> 7; st ^= st << 17; return st; }
static float unit() { return (float)(rnd() >> 40) * 0x1p-23f - 1.0f; }

static uint64_t quotients(uint64_t& n)
{
    uint64_t bad = 0;
    for (uint64_t b = 1u << 23; b < 1u << 24; b++) {
        const int v = __builtin_ctzll(b);
        const float fb = (float)b, y = 1.0f / fb;
        const uint64_t odd = b >> v;
        uint64_t inv = odd;
        for (int i = 0; i < 5; i++) inv *= 2 - odd * inv;
        /* a 2^k = b m + s, m odd of 25 bits */
        for (int64_t s = -5; s <= 5; s++) {
            if (!s || (s & ((1ll << v) - 1))) continue;
            for (int k = 24; k <= 25; k++) {
                const uint64_t mod = 1ull << (k - v);
                for (uint64_t m = (uint64_t)-(s >> v) * inv & (mod - 1); m < 1u << 25; m += mod) {
                    const uint64_t p = b * m + s, a = p >> k;
                    if (m < 1u << 24 || !(m & 1) || (p & ((1ull << k) - 1)) || a < 1u << 23 || a >= 1u << 24) continue;
                    n++;
                    bad += exact_quot((float)a, fb, y) != (float)a / fb;
                }
            }
        }
    }
    for (int i = 0; i < 4000000; i++) {
        const float a = ldexpf(unit(), (int)(rnd() % 120) - 60), b = ldexpf(1.5f + 0.5f * unit(), (int)(rnd() % 60) - 30);
        bad += exact_quot(a, b, 1.0f / b) != a / b;
    }
    return bad;
}

static uint64_t floors()
{
    uint64_t bad = 0;
    for (int i = 0; i < 2000000; i++) {
        const uint32_t d = i < 70000 ? 1 + i : 1 + (uint32_t)(rnd() >> (33 + rnd() % 31)) % 0x7FFFFFFEu;
        const uint32_t n = i & 1 ? (uint32_t)(rnd() >> 33) : ((uint32_t)(rnd() >> 33) / d) * d - (i & 2 ? 1 : 0);
        const uint32_t m = n & 0x7FFFFFFFu;
        bad += exact_div_floor(m, exact_div_of(d)) != m / d;
    }
    return bad;
}

static int same(const tgx_m4& a, const tgx_m4& b)
{
    for (int i = 0; i < 3; i++)
        for (int c = 0; c < 4; c++) {
            const float x = a.m[4 * c + i], y = b.m[4 * c + i];
            if (!(x == y || (x != x && y != y))) return 0;
        }
    return 1;
}

static uint64_t transforms(uint64_t& plain)
{
    uint64_t bad = 0;
    for (int i = 0; i < 400000; i++) {
        tgx_m4 r = tgx_m4_identity();
        const int kind = i % 10;
        const float scale = kind == 1 ? 1e18f : kind == 2 ? 1e-14f : kind == 3 ? 37.0f : 1.0f;
        if (kind != 0)
            for (int c = 0; c < 3; c++)
                for (int a = 0; a < 3; a++) r.m[4 * c + a] = scale * unit();
        if (kind == 4) r.m[rnd() % 3] = 0.0f;
        if (kind == 5) { r.m[4] = r.m[0]; r.m[5] = r.m[1]; r.m[6] = r.m[2]; }  /* singular */
        if (kind == 6) r.m[rnd() % 16] = i & 16 ? INFINITY : NAN;
        if (kind == 7) r.m[3 + 4 * (rnd() % 3)] = unit();
        if (kind == 8) for (int a = 0; a < 3; a++) r.m[rnd() % 11] = rnd() & 1 ? 0.0f : -1.0f;
        float t[3];
        for (int a = 0; a < 3; a++) t[a] = 3000.0f * unit();
        if (kind == 9 && (i & 16)) t[rnd() % 3] = i & 32 ? INFINITY : 3e38f;
        const unsigned n[3] = {1u + (unsigned)(rnd() % 40), 1u + (unsigned)(rnd() % 40), 1u + (unsigned)(rnd() % 40)};
        const unsigned x = (unsigned)(rnd() % n[0]), y = (unsigned)(rnd() % n[1]), z = (unsigned)(rnd() % n[2]);
        const float o[3] = {8.0f * x, 8.0f * y, 8.0f * z}, h[3] = {4.0f * n[0], 4.0f * n[1], 4.0f * n[2]};
        const tgx_m4 w2c = tgx_m4_mul(tgx_m4_mul(tgx_m4_mul(tgx_m4_translate(-o[0], -o[1], -o[2]),
                                                            tgx_m4_translate(h[0], h[1], h[2])), tgx_m4_inverse(r)),
                                      tgx_m4_translate(-t[0], -t[1], -t[2]));
        const tgx_m4 c2w = tgx_m4_mul(tgx_m4_mul(tgx_m4_mul(tgx_m4_translate(t[0], t[1], t[2]), r),
                                                 tgx_m4_translate(-h[0], -h[1], -h[2])), tgx_m4_translate(o[0], o[1], o[2]));
        const tgx_m4 a = tgx_world_to_cluster(r.m, t, n, x, y, z), b = tgx_cluster_to_world(r.m, t, n, x, y, z);
        plain += tgx_m4_is_3x3(r.m) && tgx_m4_rows_finite(&a);
        bad += !same(a, w2c) + !same(b, c2w);
    }
    return bad;
}

int main()
{
    uint64_t n = 0, plain = 0;
    const uint64_t q = quotients(n), f = floors(), t = transforms(plain);
    printf("%llu %llu %llu %llu %llu\n", (unsigned long long)n, (unsigned long long)q, (unsigned long long)f,
           (unsigned long long)plain, (unsigned long long)t);
}
"""


def test_host_build(tmp_path):
    src = tmp_path / "exact.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "exact"
    subprocess.run(["g++", "-O2", "-std=c++17", "-mfma", "-ffp-contract=off", "-I", str(CSRC), str(src), "-o", str(exe)],
                   check=True)
    hard, quotients, floors, plain, transforms = map(int, subprocess.run([exe], check=True, capture_output=True,
                                                                         text=True).stdout.split())
    assert hard > 2e7 and plain > 1e5
    assert (quotients, floors, transforms) == (0, 0, 0)


@pytest.mark.gpu
def test_device_reciprocal_and_root(ctx):
    assert ctx.arith_check() == (0, 0)
