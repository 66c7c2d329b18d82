"""The trace kernel's own test for leaves that a ray leaves without a hit
(tgx_leaf_clear.h), compiled for the host, against the exact 32^3 walk
(tg_amanatides_woo.c:3-114) in the kernel's arithmetic: a leaf called clear has
a walk that meets no solid voxel's brick. Entries on, beside and beyond faces and
edges, at voxel middles and corners; directions with equal, nearly equal, tiny,
zero and large components; few, many and all bricks solid."""
import subprocess
from pathlib import Path

import tg_amd as T

CSRC = Path(T.__file__).resolve().parent / "csrc"

PROGRAM = r"""
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <algorithm>
#define __device__
static float __builtin_amdgcn_fmed3f(float a, float b, float c)
{
    if (a != a || b != b || c != c) return fminf(fminf(a, b), c);
    return std::max(std::min(a, b), std::min(std::max(a, b), c));
}
#include "tgx_leaf_clear.h"

static uint64_t st = 88172645463325252ull;
static uint64_t rnd() { st ^= st << 13; st ^= st >> 7; st ^= st << 17; return st; }
static float u01() { return (float)(rnd() >> 40) * 0x1p-24f; }
static const float MAXF = 3.402823466e+38f;

static bool touches(uint64_t bm, const float g[3], const int v0[3], const float d[3], const float td[3])
{
    float t[3];
    int v[3];
    for (int a = 0; a < 3; a++) {
        v[a] = v0[a];
        t[a] = d[a] > 0.0f ? ((float)(v[a] + 1) - g[a]) / d[a] : d[a] < 0.0f ? (g[a] - (float)v[a]) / -d[a] : MAXF;
    }
    for (int it = 0; it < 100; it++) {
        if (bm >> ((v[0] >> 3) + 4 * (v[1] >> 3) + 16 * (v[2] >> 3)) & 1u) return true;
        const int a = t[0] < t[1] ? (t[0] < t[2] ? 0 : 2) : (t[1] < t[2] ? 1 : 2);
        t[a] = t[a] + td[a];
        v[a] += d[a] > 0.0f ? 1 : d[a] < 0.0f ? -1 : 0;
        if (v[a] < 0 || v[a] > 31) return false;
    }
    return true;
}

int main()
{
    uint64_t wrong = 0, found = 0, clear = 0;
    for (int i = 0; i < 6000000; i++) {
        float d[3], g[3], td[3];
        int v[3];
        for (int a = 0; a < 3; a++) d[a] = 2.0f * u01() - 1.0f;
        const int k = rnd() % 12;
        if (k == 0) for (int a = 0; a < 3; a++) d[a] = (float)((int)(rnd() % 5) - 2) * 0.5f;
        if (k == 1) d[rnd() % 3] *= 1e-6f;
        if (k == 2) d[rnd() % 3] = 0.0f;
        if (k == 3) d[0] = d[1] * (1.0f + (float)((int)(rnd() % 9) - 4) * 0x1p-22f);
        if (k == 4) d[rnd() % 3] *= ldexpf(1.0f, -(int)(rnd() % 90));
        if (k == 5) for (int a = 0; a < 3; a++) d[a] *= 0x1p20f;
        if (k == 6) { d[rnd() % 3] = 0.0f; d[rnd() % 3] = 0.0f; }
        if (d[0] == 0.0f && d[1] == 0.0f && d[2] == 0.0f) d[0] = 1.0f;
        const int p = rnd() % 6;
        for (int a = 0; a < 3; a++) {
            g[a] = 32.0f * u01();
            if (p == 0) g[a] = floorf(g[a]);
            if (p == 1) g[a] = floorf(g[a]) + 0.5f;
            if (p == 2) g[a] = 8.0f * floorf(4.99f * u01());
        }
        /* through a face, up to a few roundings of a position beyond 4096 off it */
        const int f = rnd() % 3;
        if (rnd() & 7) g[f] = (d[f] > 0.0f ? 0.0f : 32.0f) + (float)((int)(rnd() % 7) - 3) * (rnd() & 1 ? 0x1p-11f : 1e-6f);
        /* on its way out already */
        if (p == 3) g[rnd() % 3] = rnd() & 1 ? 32.0f + 0x1p-11f : -0x1p-11f;
        for (int a = 0; a < 3; a++) {
            v[a] = (int)std::min(std::max(floorf(g[a]), 0.0f), 31.0f);
            td[a] = d[a] == 0.0f ? MAXF : 1.0f / fabsf(d[a]);
        }
        uint64_t bm = rnd();
        const int s = rnd() % 4;
        if (s < 2) bm &= rnd() & rnd();
        if (s == 0) bm &= rnd() & rnd();
        const bool c = leaf_clear(bm, g[0], g[1], g[2], v[0], v[1], v[2], d[0], d[1], d[2], td[0], td[1], td[2]);
        const bool t = touches(bm, g, v, d, td);
        wrong += c && t;
        found += c;
        clear += !t;
    }
    printf("%llu %llu %llu\n", (unsigned long long)wrong, (unsigned long long)found, (unsigned long long)clear);
}
"""


def test_clear_leaves_are_walked_without_a_hit(tmp_path):
    src = tmp_path / "clear.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "clear"
    subprocess.run(["g++", "-O2", "-std=c++17", "-mfma", "-ffp-contract=off", "-I", str(CSRC), str(src), "-o", str(exe)],
                   check=True)
    wrong, found, clear = map(int, subprocess.run([exe], check=True, capture_output=True, text=True).stdout.split())
    assert wrong == 0
    assert clear > 1_000_000 and found > 0.9 * clear
