/*
 * tgx_m4.h — 4x4 matrix and 3-vector helpers shared by host C and HIP
 * device code of the product path.
 *
 * Storage is column-major, m[4*col + row], as tg's m4 (tg_math.h:240-275).
 * Every function fixes its floating-point operation order, so that host
 * and device builds (both compiled with -ffp-contract=off, IEEE fp32
 * division and square root) produce the same bits:
 *   mul:     r(i,j) = ((a(i,0)b(0,j) + a(i,1)b(1,j)) + a(i,2)b(2,j)) + a(i,3)b(3,j)
 *            (tg_math.c:2374-2399)
 *   mulv4:   r.i = ((x m(i,0) + y m(i,1)) + z m(i,2)) + w m(i,3)
 *            (tg_math.c:2428-2438)
 *   inverse: cofactor expansion of tg_math.c:2185-2234, one fp32 division.
 */
#ifndef TGX_M4_H
#define TGX_M4_H

#if defined(__HIPCC__)
#define TGX_HD __host__ __device__ static inline
#else
#define TGX_HD static inline
#endif

typedef struct tgx_m4 { float m[16]; } tgx_m4;
typedef struct tgx_v3 { float x, y, z; } tgx_v3;
typedef struct tgx_v4 { float x, y, z, w; } tgx_v4;

#define TGX_M(mat, r, c) ((mat).m[4 * (c) + (r)])

TGX_HD tgx_v3 tgx_v3_make(float x, float y, float z) { tgx_v3 v; v.x = x; v.y = y; v.z = z; return v; }

TGX_HD tgx_m4 tgx_m4_identity(void)
{
    tgx_m4 r;
    for (int i = 0; i < 16; i++) r.m[i] = 0.0f;
    r.m[0] = 1.0f; r.m[5] = 1.0f; r.m[10] = 1.0f; r.m[15] = 1.0f;
    return r;
}

TGX_HD tgx_m4 tgx_m4_translate(float x, float y, float z)
{
    tgx_m4 r = tgx_m4_identity();
    TGX_M(r, 0, 3) = x; TGX_M(r, 1, 3) = y; TGX_M(r, 2, 3) = z;
    return r;
}

TGX_HD tgx_m4 tgx_m4_mul(tgx_m4 a, tgx_m4 b)
{
    tgx_m4 r;
    for (int c = 0; c < 4; c++) {
        for (int i = 0; i < 4; i++) {
            float s = TGX_M(a, i, 0) * TGX_M(b, 0, c);
            s = s + TGX_M(a, i, 1) * TGX_M(b, 1, c);
            s = s + TGX_M(a, i, 2) * TGX_M(b, 2, c);
            s = s + TGX_M(a, i, 3) * TGX_M(b, 3, c);
            TGX_M(r, i, c) = s;
        }
    }
    return r;
}

TGX_HD tgx_v4 tgx_m4_mulv4(tgx_m4 m, float x, float y, float z, float w)
{
    tgx_v4 r;
    r.x = x * TGX_M(m, 0, 0) + y * TGX_M(m, 0, 1) + z * TGX_M(m, 0, 2) + w * TGX_M(m, 0, 3);
    r.y = x * TGX_M(m, 1, 0) + y * TGX_M(m, 1, 1) + z * TGX_M(m, 1, 2) + w * TGX_M(m, 1, 3);
    r.z = x * TGX_M(m, 2, 0) + y * TGX_M(m, 2, 1) + z * TGX_M(m, 2, 2) + w * TGX_M(m, 2, 3);
    r.w = x * TGX_M(m, 3, 0) + y * TGX_M(m, 3, 1) + z * TGX_M(m, 3, 2) + w * TGX_M(m, 3, 3);
    return r;
}

/* Cofactor inverse with the reference's sub-determinant names and order. */
TGX_HD tgx_m4 tgx_m4_inverse(tgx_m4 a)
{
#define A(r, c) TGX_M(a, r, c)
    const float m2323 = A(2,2) * A(3,3) - A(2,3) * A(3,2);
    const float m1323 = A(2,1) * A(3,3) - A(2,3) * A(3,1);
    const float m1223 = A(2,1) * A(3,2) - A(2,2) * A(3,1);
    const float m0323 = A(2,0) * A(3,3) - A(2,3) * A(3,0);
    const float m0223 = A(2,0) * A(3,2) - A(2,2) * A(3,0);
    const float m0123 = A(2,0) * A(3,1) - A(2,1) * A(3,0);
    const float m2313 = A(1,2) * A(3,3) - A(1,3) * A(3,2);
    const float m1313 = A(1,1) * A(3,3) - A(1,3) * A(3,1);
    const float m1213 = A(1,1) * A(3,2) - A(1,2) * A(3,1);
    const float m2312 = A(1,2) * A(2,3) - A(1,3) * A(2,2);
    const float m1312 = A(1,1) * A(2,3) - A(1,3) * A(2,1);
    const float m1212 = A(1,1) * A(2,2) - A(1,2) * A(2,1);
    const float m0313 = A(1,0) * A(3,3) - A(1,3) * A(3,0);
    const float m0213 = A(1,0) * A(3,2) - A(1,2) * A(3,0);
    const float m0312 = A(1,0) * A(2,3) - A(1,3) * A(2,0);
    const float m0212 = A(1,0) * A(2,2) - A(1,2) * A(2,0);
    const float m0113 = A(1,0) * A(3,1) - A(1,1) * A(3,0);
    const float m0112 = A(1,0) * A(2,1) - A(1,1) * A(2,0);

    const float det = 1.0f / (
        A(0,0) * (A(1,1) * m2323 - A(1,2) * m1323 + A(1,3) * m1223) -
        A(0,1) * (A(1,0) * m2323 - A(1,2) * m0323 + A(1,3) * m0223) +
        A(0,2) * (A(1,0) * m1323 - A(1,1) * m0323 + A(1,3) * m0123) -
        A(0,3) * (A(1,0) * m1223 - A(1,1) * m0223 + A(1,2) * m0123));

    tgx_m4 r;
    TGX_M(r,0,0) = det *  (A(1,1) * m2323 - A(1,2) * m1323 + A(1,3) * m1223);
    TGX_M(r,0,1) = det * -(A(0,1) * m2323 - A(0,2) * m1323 + A(0,3) * m1223);
    TGX_M(r,0,2) = det *  (A(0,1) * m2313 - A(0,2) * m1313 + A(0,3) * m1213);
    TGX_M(r,0,3) = det * -(A(0,1) * m2312 - A(0,2) * m1312 + A(0,3) * m1212);
    TGX_M(r,1,0) = det * -(A(1,0) * m2323 - A(1,2) * m0323 + A(1,3) * m0223);
    TGX_M(r,1,1) = det *  (A(0,0) * m2323 - A(0,2) * m0323 + A(0,3) * m0223);
    TGX_M(r,1,2) = det * -(A(0,0) * m2313 - A(0,2) * m0313 + A(0,3) * m0213);
    TGX_M(r,1,3) = det *  (A(0,0) * m2312 - A(0,2) * m0312 + A(0,3) * m0212);
    TGX_M(r,2,0) = det *  (A(1,0) * m1323 - A(1,1) * m0323 + A(1,3) * m0123);
    TGX_M(r,2,1) = det * -(A(0,0) * m1323 - A(0,1) * m0323 + A(0,3) * m0123);
    TGX_M(r,2,2) = det *  (A(0,0) * m1313 - A(0,1) * m0313 + A(0,3) * m0113);
    TGX_M(r,2,3) = det * -(A(0,0) * m1312 - A(0,1) * m0312 + A(0,3) * m0112);
    TGX_M(r,3,0) = det * -(A(1,0) * m1223 - A(1,1) * m0223 + A(1,2) * m0123);
    TGX_M(r,3,1) = det *  (A(0,0) * m1223 - A(0,1) * m0223 + A(0,2) * m0123);
    TGX_M(r,3,2) = det * -(A(0,0) * m1213 - A(0,1) * m0213 + A(0,2) * m0113);
    TGX_M(r,3,3) = det *  (A(0,0) * m1212 - A(0,1) * m0212 + A(0,2) * m0112);
#undef A
    return r;
}

/* Rows 0..2 of an affine matrix with bottom row (0, 0, 0, w). */
TGX_HD tgx_m4 tgx_m4_rows(float m00, float m01, float m02, float m03, float m10, float m11, float m12, float m13,
                          float m20, float m21, float m22, float m23, float w)
{
    tgx_m4 r;
    TGX_M(r,0,0) = m00; TGX_M(r,0,1) = m01; TGX_M(r,0,2) = m02; TGX_M(r,0,3) = m03;
    TGX_M(r,1,0) = m10; TGX_M(r,1,1) = m11; TGX_M(r,1,2) = m12; TGX_M(r,1,3) = m13;
    TGX_M(r,2,0) = m20; TGX_M(r,2,1) = m21; TGX_M(r,2,2) = m22; TGX_M(r,2,3) = m23;
    TGX_M(r,3,0) = 0.0f; TGX_M(r,3,1) = 0.0f; TGX_M(r,3,2) = 0.0f; TGX_M(r,3,3) = w;
    return r;
}

/* Sum of the magnitudes of rows 0..2 is finite: so is every element. */
TGX_HD int tgx_m4_rows_finite(const tgx_m4* r)
{
    float s = 0.0f;
    for (int i = 0; i < 3; i++)
        for (int c = 0; c < 4; c++) s = s + (TGX_M(*r, i, c) < 0.0f ? -TGX_M(*r, i, c) : TGX_M(*r, i, c));
    return s <= 3.402823466e+38f;
}

/* An object's rotation that is a 3x3 matrix in a 4x4 one, as every rotation
 * and scaling is. The two transforms below then leave out the products with
 * the zeros and ones of the translations and of this matrix, about 500
 * operations a cluster or pixel down to 80: for finite elements they add +-0
 * to the sums that are left or multiply them by one, so each element keeps its
 * value (a zero may change its sign). Where an element is not finite, the
 * products are taken, as 0 times it is NaN. */
TGX_HD int tgx_m4_is_3x3(const float m[16])
{
    return m[3] == 0.0f && m[7] == 0.0f && m[11] == 0.0f && m[12] == 0.0f && m[13] == 0.0f && m[14] == 0.0f &&
           m[15] == 1.0f;
}

/* World -> cluster space of cluster (rx, ry, rz) of an object with
 * n clusters per axis: T(-offset) * T(+half) * inverse(R) * T(-t),
 * associated left to right (visibility.frag:57-62,
 * tg_sparse_voxel_octree.c:53-57). The cluster then spans [0,8]^3. */
TGX_HD tgx_m4 tgx_world_to_cluster(const float rotation[16], const float translation[3],
                                   const unsigned n[3], unsigned rx, unsigned ry, unsigned rz)
{
    tgx_m4 rot;
    for (int i = 0; i < 16; i++) rot.m[i] = rotation[i];
    const float offx = (float)(rx * 8u), offy = (float)(ry * 8u), offz = (float)(rz * 8u);
    const float hx = 4.0f * (float)n[0], hy = 4.0f * (float)n[1], hz = 4.0f * (float)n[2];
    if (tgx_m4_is_3x3(rotation)) {
#define A(r, c) TGX_M(rot, r, c)
        const float m12 = A(1,1) * A(2,2) - A(1,2) * A(2,1);
        const float m02 = A(1,0) * A(2,2) - A(1,2) * A(2,0);
        const float m01 = A(1,0) * A(2,1) - A(1,1) * A(2,0);
        const float d = A(0,0) * m12 - A(0,1) * m02 + A(0,2) * m01;
        const float det = 1.0f / d;
        const float r00 = det * m12, r01 = det * -(A(0,1) * A(2,2) - A(0,2) * A(2,1)),
                    r02 = det * (A(0,1) * A(1,2) - A(0,2) * A(1,1));
        const float r10 = det * -m02, r11 = det * (A(0,0) * A(2,2) - A(0,2) * A(2,0)),
                    r12 = det * -(A(0,0) * A(1,2) - A(0,2) * A(1,0));
        const float r20 = det * m01, r21 = det * -(A(0,0) * A(2,1) - A(0,1) * A(2,0)),
                    r22 = det * (A(0,0) * A(1,1) - A(0,1) * A(1,0));
        const float w = det * d; /* 1 to within a rounding */
#undef A
        const float tx = -translation[0], ty = -translation[1], tz = -translation[2];
        const tgx_m4 r = tgx_m4_rows(r00, r01, r02, r00 * tx + r01 * ty + r02 * tz + (hx + -offx) * w,
                                     r10, r11, r12, r10 * tx + r11 * ty + r12 * tz + (hy + -offy) * w,
                                     r20, r21, r22, r20 * tx + r21 * ty + r22 * tz + (hz + -offz) * w, w);
        if (tgx_m4_rows_finite(&r)) return r;
    }
    const tgx_m4 m0 = tgx_m4_translate(-translation[0], -translation[1], -translation[2]);
    const tgx_m4 m1 = tgx_m4_inverse(rot);
    const tgx_m4 m2 = tgx_m4_translate(hx, hy, hz);
    const tgx_m4 m3 = tgx_m4_translate(-offx, -offy, -offz);
    return tgx_m4_mul(tgx_m4_mul(tgx_m4_mul(m3, m2), m1), m0);
}

/* Cluster -> world space: T(t) * R * T(-half) * T(+offset), associated
 * left to right (tg_sparse_voxel_octree.c:92-97). */
TGX_HD tgx_m4 tgx_cluster_to_world(const float rotation[16], const float translation[3],
                                   const unsigned n[3], unsigned rx, unsigned ry, unsigned rz)
{
    tgx_m4 rot;
    for (int i = 0; i < 16; i++) rot.m[i] = rotation[i];
    const float offx = (float)(rx * 8u), offy = (float)(ry * 8u), offz = (float)(rz * 8u);
    const float hx = (float)n[0] * 4.0f, hy = (float)n[1] * 4.0f, hz = (float)n[2] * 4.0f;
    if (tgx_m4_is_3x3(rotation)) {
        float c[3];
        for (int i = 0; i < 3; i++) {
            const float r0 = TGX_M(rot, i, 0), r1 = TGX_M(rot, i, 1), r2 = TGX_M(rot, i, 2);
            c[i] = r0 * -hx + r1 * -hy + r2 * -hz + translation[i];
            c[i] = r0 * offx + r1 * offy + r2 * offz + c[i];
        }
        const tgx_m4 r = tgx_m4_rows(TGX_M(rot, 0, 0), TGX_M(rot, 0, 1), TGX_M(rot, 0, 2), c[0],
                                     TGX_M(rot, 1, 0), TGX_M(rot, 1, 1), TGX_M(rot, 1, 2), c[1],
                                     TGX_M(rot, 2, 0), TGX_M(rot, 2, 1), TGX_M(rot, 2, 2), c[2], 1.0f);
        if (tgx_m4_rows_finite(&r)) return r;
    }
    const tgx_m4 m1 = tgx_m4_translate(offx, offy, offz);
    const tgx_m4 m2 = tgx_m4_translate(-hx, -hy, -hz);
    const tgx_m4 m4_ = tgx_m4_translate(translation[0], translation[1], translation[2]);
    return tgx_m4_mul(tgx_m4_mul(tgx_m4_mul(m4_, rot), m2), m1);
}

#endif /* TGX_M4_H */
