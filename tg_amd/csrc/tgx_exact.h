/*
 * tgx_exact.h — correctly rounded fp32 reciprocals, square roots and
 * quotients in fewer operations than the compiler's IEEE expansions, for
 * operands whose range the caller has checked.
 *
 * The expansions spend 11 to 15 operations a piece, most of them on scaling
 * for operands near the ends of the exponent range; kernels that divide a ray's
 * coordinates by its direction spent half of their issue slots there (1080p:
 * visibility traversal 120 -> 81 us, shading 46 -> 31, GI surfaces 43 -> 34 with
 * these and the shorter cluster transforms). Here:
 *
 *   exact_recip  fl(1 / d), 2^-100 <= |d| <= 2^100: v_rcp_f32 and one Newton
 *                step. Compared with the IEEE division over every float of
 *                that range (tgx_arith_check).
 *   exact_root   fl(sqrt(x)), 2^-100 <= x <= 2^100: v_rsq_f32 and one
 *                correction by the remainder; compared likewise.
 *   exact_quot   fl(a / b) from y = fl(1 / b): a y is within 1.5 ulp, and one
 *                correction by the remainder rounds right (P. Markstein,
 *                "Computation of elementary functions on the IBM RISC
 *                System/6000 processor", 1990). The corrected
 *                value's distance from a / b is below 2^-22 ulp, so only
 *                quotients that close to the middle of two floats could go
 *                wrong; all 9.3e7 pairs of 24-bit significands with
 *                |a 2^k - b m| <= 16 for such a middle m (three times the
 *                bound) were tried on the CPU and round right. a is 0 (a zero
 *                quotient may lose its sign) or so large that the quotient is
 *                normal and the remainder, a multiple of a's last bit times
 *                2^-24, is one of 2^-149: |a| >= 2^-101 and |a / b| >= 2^-101.
 */
#ifndef TGX_EXACT_H
#define TGX_EXACT_H

__device__ static inline float exact_recip(float d)
{
    const float y = __builtin_amdgcn_rcpf(d);
    return fmaf(fmaf(-d, y, 1.0f), y, y);
}

__device__ static inline float exact_root(float x)
{
    const float y = __builtin_amdgcn_rsqf(x);
    const float g = x * y;
    return fmaf(fmaf(-g, g, x), 0.5f * y, g);
}

__device__ static inline float exact_quot(float a, float b, float y)
{
    const float q = a * y;
    return fmaf(fmaf(-q, b, a), y, q);
}

/* True when each of x, y, z is 0 or lo <= |v| <= hi (NaN: false). lo, hi > 0.
 * Twice the bits drop the sign; 0 less one is above every float. */
__device__ static inline bool exact_range3(float x, float y, float z, float lo, float hi)
{
    const uint32_t a = (__float_as_uint(x) << 1) - 1u, b = (__float_as_uint(y) << 1) - 1u,
                   c = (__float_as_uint(z) << 1) - 1u;
    const uint32_t mn = min(min(a, b), c);
    const float mx = fmaxf(fmaxf(fabsf(x), fabsf(y)), fabsf(z));
    return mn >= (__float_as_uint(lo) << 1) - 1u && mx <= hi && x == x && y == y && z == z;
}

/* v / |v| of tg's normalisations: three IEEE quotients by the IEEE root of
 * (x x + y y) + z z. */
__device__ static inline void exact_normalize3(float& x, float& y, float& z)
{
    const float s = x * x + y * y + z * z;
    /* s in range bounds the components from above and excludes NaN */
    const uint32_t a = (__float_as_uint(x) << 1) - 1u, b = (__float_as_uint(y) << 1) - 1u,
                   c = (__float_as_uint(z) << 1) - 1u;
    if (s >= 0x1p-60f && s <= 0x1p60f && min(min(a, b), c) >= (__float_as_uint(0x1p-70f) << 1) - 1u) {
        const float m = exact_root(s), r = exact_recip(m);
        x = exact_quot(x, m, r);
        y = exact_quot(y, m, r);
        z = exact_quot(z, m, r);
    } else {
        const float m = sqrtf(s);
        x = x / m;
        y = y / m;
        z = z / m;
    }
}

/* tg_intersect_ray_aabb (collide.inc:3-24) with a box of integer corners in
 * [0, 8]: near and far distance of one axis are each one quotient, its
 * numerator chosen by the direction's sign, all by the reciprocal of the axis. With
 * |o| in {0} u [2^-50, 2^30] the numerators are 0 or at least 2^-74. Other
 * operands take IEEE divisions. */
__device__ static inline bool exact_slab(float ox, float oy, float oz, float dx, float dy, float dz, float mnx,
                                         float mny, float mnz, float mxx, float mxy, float mxz, float& enter,
                                         float& exit_)
{
    float nx, ny, nz, fx, fy, fz;
    const float ax = dx > 0.0f ? mnx - ox : ox - mxx, bx = dx > 0.0f ? mxx - ox : ox - mnx;
    const float ay = dy > 0.0f ? mny - oy : oy - mxy, by = dy > 0.0f ? mxy - oy : oy - mny;
    const float az = dz > 0.0f ? mnz - oz : oz - mxz, bz = dz > 0.0f ? mxz - oz : oz - mnz;
    if (exact_range3(ox, oy, oz, 0x1p-50f, 0x1p30f) && exact_range3(dx, dy, dz, 0x1p-60f, 2.0f)) {
        const float rx = exact_recip(fabsf(dx)), ry = exact_recip(fabsf(dy)), rz = exact_recip(fabsf(dz));
        nx = exact_quot(ax, fabsf(dx), rx); fx = exact_quot(bx, fabsf(dx), rx);
        ny = exact_quot(ay, fabsf(dy), ry); fy = exact_quot(by, fabsf(dy), ry);
        nz = exact_quot(az, fabsf(dz), rz); fz = exact_quot(bz, fabsf(dz), rz);
    } else {
        nx = ax / fabsf(dx); fx = bx / fabsf(dx);
        ny = ay / fabsf(dy); fy = by / fabsf(dy);
        nz = az / fabsf(dz); fz = bz / fabsf(dz);
    }
    nx = dx == 0.0f ? -3.402823466e+38f : nx; fx = dx == 0.0f ? 3.402823466e+38f : fx;
    ny = dy == 0.0f ? -3.402823466e+38f : ny; fy = dy == 0.0f ? 3.402823466e+38f : fy;
    nz = dz == 0.0f ? -3.402823466e+38f : nz; fz = dz == 0.0f ? 3.402823466e+38f : fz;
    enter = nx > ny ? nx : ny;
    enter = enter > nz ? enter : nz;
    exit_ = fx < fy ? fx : fy;
    exit_ = exit_ < fz ? exit_ : fz;
    return exit_ > 0.0f && enter <= exit_;
}

/* floor(n / d) for n < 2^31 by one multiplication; mul 0 stands for d = 1.
 * mul = ceil(2^(31 + s) / d) with 2^s >= d exceeds the true value by less than
 * 2^s / d of a unit, so n mul / 2^(31 + s) stays below the next integer. */
struct exact_div {
    uint32_t mul, shift;
};

static inline exact_div exact_div_of(uint32_t d)
{
    exact_div r = {0u, 0u};
    if (d <= 1u) return r;
    uint32_t s = 1u;
    while (s < 31u && (1ull << s) < d) s++;
    r.mul = (uint32_t)(((1ull << (31u + s)) + d - 1u) / d);
    r.shift = s - 1u;
    return r;
}

__device__ static inline uint32_t exact_div_floor(uint32_t n, exact_div d)
{
    return d.mul ? __umulhi(n, d.mul) >> d.shift : n;
}

#endif /* TGX_EXACT_H */
