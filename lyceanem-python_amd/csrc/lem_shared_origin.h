// lem_shared_origin.h -- tests that say which triangles a ray from a known origin
// cannot hit, for the dense visibility kernel: rays of one origin share them.
// Plain per-element code, so the CPU checks compile it too (LEM_HOST_BUILD).
//
// With t = o - v0 and q = t x e1
// the predicate's dot products are linear in the ray's direction d with
// coefficients that belong to the triangle alone:
//   A = d . (e2 x e1),  du = d . (e2 x t),  dv = d . q,  dt = e2 . q.
// dt does not depend on the ray at all, and a hit needs t = dt / A > 0, so A
// has dt's sign: the three vectors are multiplied by it (a triangle with
// dt == 0 is never hit from o).  A ray can be hit only if
//   du >= 0,  dv >= 0,  A - du - dv >= 0   and  |dt| < dist A,
// each up to rounding.  The loop tests just that -- 16 operations a ray and
// triangle instead of the predicate's about 57 -- and runs the predicate
// itself, as written, on what is left, in table order.
// Margins, with E = 2^-24 and one-norms (|d_i| <= 1): the predicate's du is at
// most 5.1 E |t||e2| from d . (e2 x t), the loop's at most 10.1 E, and likewise
// for A (|e1||e2|) and dv (|t||e1|); the predicate also takes du + dv <=
// A (1 + 2.2e-6) (its band around U + V = 1), 37 E |e1||e2|, and the two
// differences of the test add 9 E |e1||e2|.  M = 64 E |e1||e2| + 16 E |t|(|e1| + |e2|)
// and 24 E |e1||e2| for A in the distance test cover them.  Overflow makes M
// infinite and a NaN fails every comparison: both leave the triangle to the
// predicate.
//
#pragma once

#include "lem_device.h"

namespace lem {

// Largest value of n . d over the box.
LEM_DEV float box_max(float nx, float ny, float nz, float cx, float cy, float cz,
                                         float hx, float hy, float hz)
{
    const float m = __builtin_fmaf(nz, cz, __builtin_fmaf(ny, cy, nx * cx));
    return __builtin_fmaf(fabsf(nz), hz, __builtin_fmaf(fabsf(ny), hy,
                                                        __builtin_fmaf(fabsf(nx), hx, m)));
}

// n . d, fused.
LEM_DEV float dot_fma(const Ray &r, const float4 &n)
{
    return __builtin_fmaf(r.dz, n.z, __builtin_fmaf(r.dy, n.y, r.dx * n.x));
}

// The linear tests of one triangle from origin o (k_visibility_dense): (a, M),
// (u, 24 E |e1||e2|), (v, |dt|), and the ball of directions outside which no ray
// from o passes them.
//
// The ball.  Let d pass: du, dv, w = A - du - dv >= -M.  (i) A >= 32 M: the point
// where the ray meets the plane has barycentric coordinates above -1/32, so it
// lies in the triangle scaled by 1 + 3/32 and d in the cone of the sphere of
// radius 1.1 rho around the centroid (rho: the vertices' largest distance from
// it).  (ii) A < 32 M: then |du|, |dv| <= 34 M, and as u, v are perpendicular to t
// with |u x v| = |t||dt|, d is within b = 34 M (|u| + |v|) / (|t||dt|) of the line
// through o and v0; on v0's far side of o A would be below -3 M if |dt| >
// |t| (3 M + |a| b), so d is within b of v0, a point of the sphere.  The ball is
// the cone widened by 0.03 where b <= 0.02 and |dt| >= 2 |t| (3 M + |a| b); a
// triangle seen more nearly edge on, or from inside its sphere, has none
// (radius 4).
template <int SEM>
LEM_DEV void shared_origin_tests(const Tri &t, float ox, float oy, float oz,
                                                    float4 &ca, float4 &cu, float4 &cv,
                                                    float4 &ball)
{
    const float tx = ox - t.v0x, ty = oy - t.v0y, tz = oz - t.v0z;
    const float qx = ty * t.e1z - tz * t.e1y;
    const float qy = tz * t.e1x - tx * t.e1z;
    const float qz = tx * t.e1y - ty * t.e1x;
    float dt = t.e2x * qx + t.e2y * qy;
    dt = dt + t.e2z * qz;
    // the native predicate also needs A > 0
    if (!(SEM == 0 ? fabsf(dt) > 0.0f : dt > 0.0f))
        return;
    const float E = 5.9604645e-8f;
    const float sg = __builtin_copysignf(1.0f, dt);
    const float n1 = fabsf(t.e1x) + fabsf(t.e1y) + fabsf(t.e1z);
    const float n2 = fabsf(t.e2x) + fabsf(t.e2y) + fabsf(t.e2z);
    const float nt = fabsf(tx) + fabsf(ty) + fabsf(tz);
    const float M = E * (64.0f * n1 * n2 + 16.0f * nt * (n1 + n2)) + 1e-30f;
    ca = make_float4(sg * (t.e2y * t.e1z - t.e2z * t.e1y), sg * (t.e2z * t.e1x - t.e2x * t.e1z),
                     sg * (t.e2x * t.e1y - t.e2y * t.e1x), M);
    cu = make_float4(sg * (t.e2y * tz - t.e2z * ty), sg * (t.e2z * tx - t.e2x * tz),
                     sg * (t.e2x * ty - t.e2y * tx), 24.0f * E * n1 * n2 + 1e-30f);
    cv = make_float4(sg * qx, sg * qy, sg * qz, fabsf(dt));
    const float THIRD = 0.33333334f;
    const float gx = (t.e1x + t.e2x) * THIRD, gy = (t.e1y + t.e2y) * THIRD,
                gz = (t.e1z + t.e2z) * THIRD;
    const float hx = t.e1x - gx, hy = t.e1y - gy, hz = t.e1z - gz;
    const float kx = t.e2x - gx, ky = t.e2y - gy, kz = t.e2z - gz;
    const float rho2 = fmaxf(gx * gx + gy * gy + gz * gz,
                             fmaxf(hx * hx + hy * hy + hz * hz, kx * kx + ky * ky + kz * kz));
    const float px = gx - tx, py = gy - ty, pz = gz - tz;
    const float D2 = px * px + py * py + pz * pz;
    const float x2 = 1.22f * rho2 * rcpf_estimate(D2);  // sin^2 of the cone's half angle
    // one-norms bound |t|, |u|, |v| and |a| from above
    const float na = fabsf(ca.x) + fabsf(ca.y) + fabsf(ca.z);
    const float nu = fabsf(cu.x) + fabsf(cu.y) + fabsf(cu.z);
    const float nv = fabsf(cv.x) + fabsf(cv.y) + fabsf(cv.z);
    const float t2 = 1.001f * sqrtf_estimate(tx * tx + ty * ty + tz * tz);
    const float b = 35.0f * M * (nu + nv) * rcpf_estimate(t2 * fabsf(dt));
    if (x2 < 0.98f && b <= 0.02f && fabsf(dt) >= 2.0f * t2 * (3.0f * M + na * b)) {
        const float inv = rcpf_estimate(sqrtf_estimate(D2));
        ball = make_float4(px * inv, py * inv, pz * inv,
                           sqrtf_estimate(2.0f - 2.0f * sqrtf_estimate(1.0f - x2)) + 0.031f);
    }
}

// True when the ray cannot hit the triangle of (a, u, v) nearer than dist.
LEM_DEV bool shared_origin_out(const Ray &r, float dist, const float4 &a, const float4 &u,
                               const float4 &v)
{
    const float A = dot_fma(r, a), du = dot_fma(r, u), dv = dot_fma(r, v);
    const float w = (A - du) - dv;
    return (fminf(fminf(du, dv), w) < -a.w) | (__builtin_fmaf(dist, A + u.w, -v.w) < 0.0f);
}

// True when no ray with a direction in the box (centre c, half widths h) can hit it.
LEM_DEV bool shared_origin_box_out(const float4 &a, const float4 &u, const float4 &v,
                                   const float4 &ball, float cx, float cy, float cz, float hx,
                                   float hy, float hz)
{
    const float mu = box_max(u.x, u.y, u.z, cx, cy, cz, hx, hy, hz);
    const float mv = box_max(v.x, v.y, v.z, cx, cy, cz, hx, hy, hz);
    const float mw = box_max((a.x - u.x) - v.x, (a.y - u.y) - v.y, (a.z - u.z) - v.z, cx, cy, cz,
                             hx, hy, hz);
    return (fminf(fminf(mu, mv), mw) < -4.0f * a.w) | (fabsf(ball.x - cx) > hx + ball.w) |
           (fabsf(ball.y - cy) > hy + ball.w) | (fabsf(ball.z - cz) > hz + ball.w);
}

}  // namespace lem
