// lem_beam_walk.h -- the walk of a wavefront's 64 rays through the grid as one
// beam (lem_grid.hip's persistent traversal).
//
// The 64 rays share one end, P; their other ends lie in the box [P + A, P + B].
// At the fraction u of the way every ray is inside P + u [A, B], so the macro
// blocks that any ray can meet are found once for all 64, a slab of blocks a lane
// (beam_slab, beam_block), instead of being stepped through by each ray; the rays
// then visit the blocks left over together, so that the lanes of a wavefront read
// the same cells, and a ray walks only the cells inside the content box of a block
// it meets (block_walk).  Like lem_grid_walk.h this is plain per-lane code that also
// compiles as host C++.
#pragma once

#include "lem_grid_walk.h"

namespace lem {

constexpr int BEAM_NA = 8, BEAM_NB = 4;  // most blocks of a slab, on the two other axes
constexpr int BEAM_MAX = 16;             // and in all

// On one axis, u of the lines P + u A = x and P + u B = x as x iA + c: an upper
// bound of u (cu) or a lower one (cl), whichever P + u A <= x (P + u B >= x) makes it;
// the other constant is out of the way.  The beam's margin is in the constants.
struct BeamAxis {
    float iA, cAu, cAl, iB, cBu, cBl;
};

// reciprocal of x away from zero (a bound of zero width becomes one of 1e-18); its
// error of an ulp is in the margin
LEM_DEV float beam_recip(float x)
{
    return rcpf_estimate(fabsf(x) > 1e-18f ? x : __builtin_copysignf(1e-18f, x));
}

LEM_DEV BeamAxis beam_axis(float p, float a, float b, float mrg)
{
    constexpr float BIG = 1e30f;
    BeamAxis k;
    k.iA = beam_recip(a);
    k.iB = beam_recip(b);
    const float cA = (mrg - p) * k.iA, cB = -(mrg + p) * k.iB;
    k.cAu = __builtin_signbit(a) ? BIG : cA;
    k.cAl = __builtin_signbit(a) ? cA : -BIG;
    k.cBu = __builtin_signbit(b) ? cB : BIG;
    k.cBl = __builtin_signbit(b) ? -BIG : cB;
    return k;
}

// The fractions u for which P + u A <= hi and P + u B >= lo narrow [u0, u1].
LEM_DEV void beam_clip(const BeamAxis &k, float lo, float hi, float &u0, float &u1)
{
    u1 = fminf(u1, fminf(__builtin_fmaf(hi, k.iA, k.cAu), __builtin_fmaf(lo, k.iB, k.cBu)));
    u0 = fmaxf(u0, fmaxf(__builtin_fmaf(hi, k.iA, k.cAl), __builtin_fmaf(lo, k.iB, k.cBl)));
}

struct Beam {
    // axis m (the one with the most slabs), then the other two, a and b
    float pa, pb, aa, ab, ba, bb;
    float lom, sm;             // grid origin and block extent on m
    float ia, ib;              // blocks per unit on a and b
    BeamAxis m;
    float mrg;                 // covers the rounding of every test below
    int axis;                  // m
    int na, nb;                // blocks on a and b
    int first, step, slabs;    // slabs in the rays' direction
};

// What covers the rounding of every test of a beam: each is a handful of float32
// operations on values up to the points' and their differences.
LEM_DEV float beam_margin(const GridDev &G, float px, float py, float pz, float lox, float loy,
                          float loz, float hix, float hiy, float hiz)
{
    const float far = fmaxf(fmaxf(fmaxf(fabsf(lox - px), fabsf(hix - px)),
                                  fmaxf(fabsf(loy - py), fabsf(hiy - py))),
                            fmaxf(fabsf(loz - pz), fabsf(hiz - pz)));
    const float at = fmaxf(fmaxf(fabsf(px), fabsf(py)), fabsf(pz));
    return 2.0f * G.eps + 1e-6f * (far + at);
}

// The beam from P to the box [lo, hi]; from_p: the rays start at P.  False: too
// wide for it, or not finite (the rays then walk one by one).
LEM_DEV bool beam_of(const GridDev &G, float px, float py, float pz, float lox, float loy, float loz,
                     float hix, float hiy, float hiz, bool from_p, Beam &b)
{
    // read before they are chosen among (a choice of members would keep G in memory)
    const float glx = G.lox, gly = G.loy, glz = G.loz, gcx = G.cx, gcy = G.cy, gcz = G.cz;
    const int gmx = G.mx, gmy = G.my, gmz = G.mz;
    const float ax = lox - px, ay = loy - py, az = loz - pz;
    const float bx = hix - px, by = hiy - py, bz = hiz - pz;
    const float mrg = beam_margin(G, px, py, pz, lox, loy, loz, hix, hiy, hiz);
    if (!(mrg < 1e30f))
        return false;
    // blocks per unit (cells per unit times a power of two) and the ends in blocks
    const float inv = __builtin_bit_cast(float, (127 - G.mshift) << 23);
    const float ix = G.icx * inv, iy = G.icy * inv, iz = G.icz * inv;
    const float gx = (float)(gmx - 1), gy = (float)(gmy - 1), gz = (float)(gmz - 1);
    const float f0x = fmaxf(floorf((fminf(px, lox) - mrg - glx) * ix), 0.0f),
                f0y = fmaxf(floorf((fminf(py, loy) - mrg - gly) * iy), 0.0f),
                f0z = fmaxf(floorf((fminf(pz, loz) - mrg - glz) * iz), 0.0f);
    const float nx = fminf(floorf((fmaxf(px, hix) + mrg - glx) * ix), gx) - f0x,
                ny = fminf(floorf((fmaxf(py, hiy) + mrg - gly) * iy), gy) - f0y,
                nz = fminf(floorf((fmaxf(pz, hiz) + mrg - glz) * iz), gz) - f0z;
    b.mrg = mrg;
    b.slabs = 0;
    b.axis = b.first = b.step = 0;
    if (fminf(nx, fminf(ny, nz)) < 0.0f)
        return true;  // outside the grid
    const bool mx = nx >= ny && nx >= nz, my = !mx && ny >= nz, mz = !mx && !my;
    b.axis = mx ? 0 : (my ? 1 : 2);
    // the others of x: y, z; of y: x, z; of z: x, y
    b.pa = mx ? py : px; b.aa = mx ? ay : ax; b.ba = mx ? by : bx; b.ia = mx ? iy : ix;
    b.pb = mz ? py : pz; b.ab = mz ? ay : az; b.bb = mz ? by : bz; b.ib = mz ? iy : iz;
    b.na = mx ? gmy : gmx;
    b.nb = mz ? gmy : gmz;
    // the wide end, in blocks
    const float wa = fminf((b.ba - b.aa + 2.0f * mrg) * b.ia, (float)b.na),
                wb = fminf((b.bb - b.ab + 2.0f * mrg) * b.ib, (float)b.nb);
    if (!(wa * wb <= (float)BEAM_MAX))
        return false;
    b.pa -= mx ? gly : glx;
    b.pb -= mz ? gly : glz;
    const float am = mx ? ax : (my ? ay : az), bm = mx ? bx : (my ? by : bz);
    b.m = beam_axis(mx ? px : (my ? py : pz), am, bm, mrg);
    b.lom = mx ? glx : (my ? gly : glz);
    b.sm = (mx ? gcx : (my ? gcy : gcz)) * (float)(1 << G.mshift);
    const int j0 = (int)(mx ? f0x : (my ? f0y : f0z));
    b.slabs = (int)(mx ? nx : (my ? ny : nz)) + 1;
    const bool up = (am + bm >= 0.0f) == from_p;
    b.first = up ? j0 : j0 + b.slabs - 1;
    b.step = up ? 1 : -1;
    return true;
}

// The blocks [a0, a0 + na) x [b0, b0 + nb) the beam meets in slab j of its axis;
// returns na nb (0: none).
LEM_DEV int beam_slab(const Beam &b, int j, int &a0, int &na, int &b0, int &nb)
{
    float u0 = 0.0f, u1 = 1.0f;
    const float lo = __builtin_fmaf(b.sm, (float)j, b.lom);
    beam_clip(b.m, lo, lo + b.sm, u0, u1);
    a0 = b0 = na = nb = 0;
    if (!(u0 <= u1))
        return 0;
    const float a_lo = floorf((fminf(u0 * b.aa, u1 * b.aa) + (b.pa - b.mrg)) * b.ia);
    const float a_hi = floorf((fmaxf(u0 * b.ba, u1 * b.ba) + (b.pa + b.mrg)) * b.ia);
    const float b_lo = floorf((fminf(u0 * b.ab, u1 * b.ab) + (b.pb - b.mrg)) * b.ib);
    const float b_hi = floorf((fmaxf(u0 * b.bb, u1 * b.bb) + (b.pb + b.mrg)) * b.ib);
    a0 = (int)fminf(fmaxf(a_lo, 0.0f), 2e6f);
    b0 = (int)fminf(fmaxf(b_lo, 0.0f), 2e6f);
    na = (int)fminf(fmaxf(a_hi, -1.0f), (float)(b.na - 1)) + 1 - a0;
    nb = (int)fminf(fmaxf(b_hi, -1.0f), (float)(b.nb - 1)) + 1 - b0;
    return na > 0 && nb > 0 ? na * nb : 0;
}

// block (on m, a, b) -> (x, y, z)
LEM_DEV void beam_block_at(int axis, int m, int a, int b, int &jx, int &jy, int &jz)
{
    jx = axis == 0 ? m : a;
    jy = axis == 1 ? m : (axis == 0 ? a : b);
    jz = axis == 2 ? m : b;
}

// The blocks of slab j whose content (smq: quantised boxes) the beam meets, as a mask
// (bit 8 ib + ia).
LEM_DEV uint32_t beam_mask(const GridDev &G, const MacroTab &smq, int axis, const BeamAxis &x,
                           const BeamAxis &y, const BeamAxis &z, int j, int a0, int na, int b0,
                           int n)
{
    uint32_t mask = 0;
    int ia = 0, bit = 0, ib = 0;
    for (int i = 0; i < n; ++i) {
        int jx, jy, jz;
        beam_block_at(axis, j, a0 + ia, b0 + ib, jx, jy, jz);
        const uint2 qv = smq[(jz * G.my + jy) * G.mx + jx];
        const float ox = macro_origin(G.qlx, G.cx, jx, G.mshift),
                    oy = macro_origin(G.qly, G.cy, jy, G.mshift),
                    oz = macro_origin(G.qlz, G.cz, jz, G.mshift);
        float u0 = 0.0f, u1 = 1.0f;
        beam_clip(x, __builtin_fmaf((float)(qv.x & 255u), G.qx, ox),
                  __builtin_fmaf((float)(qv.x >> 24), G.qx, ox), u0, u1);
        beam_clip(y, __builtin_fmaf((float)((qv.x >> 8) & 255u), G.qy, oy),
                  __builtin_fmaf((float)(qv.y & 255u), G.qy, oy), u0, u1);
        beam_clip(z, __builtin_fmaf((float)((qv.x >> 16) & 255u), G.qz, oz),
                  __builtin_fmaf((float)((qv.y >> 8) & 255u), G.qz, oz), u0, u1);
        if (((qv.x & 255u) <= (qv.x >> 24)) & (u0 <= u1))
            mask |= 1u << (bit + ia);
        if (++ia == na) {
            ia = 0;
            ++ib;
            bit += BEAM_NA;
        }
    }
    return mask;
}

// A pencil: a beam so narrow that its rays cross the same cells.  Then the cells are
// found for all rays at once too, and every ray is tested with every triangle of them.
// Sub-blocks of 4 x 4 x 4 cells, one cell a lane.

// Sides of a box, in cells: their largest product.
LEM_DEV float box_section(const GridDev &G, float dx, float dy, float dz, float &longest)
{
    const float x = dx * G.icx, y = dy * G.icy, z = dz * G.icz;
    longest = fmaxf(x, fmaxf(y, z));
    return fmaxf(x * y, fmaxf(x * z, y * z));
}

// Whether the rays to the points of a box are a pencil.  The points of a line span a fan
// of cells, not one, and the wider it is the fewer of its rays come near a triangle:
// at most 8 cells, half as many in a full grid, and half or a quarter of that where
// blocks are larger than 4 x 4 x 4 cells.  As pencils and one by one, us, from a line of
// 1,024 points (8 cells: 256) to 4,000, cells a word:
//                                1            2            4            8
//   volume of 5,000, blocks of 4   324, 445     326, 467     353, 491     301, 357
//   50,000 (full)                  623, 762     776, 896   1,045, 1,124   578, 579
//   150,000 (full)               1,069, 1,101 1,369, 1,372 1,853, 1,791   854, 822
//   500,000 (full), blocks of 8  1,049, 1,036 1,399, 1,269 2,055, 1,590 1,252, 797
//   terrain of 10^6, blocks of 8   336, 406     333, 433     382, 456     383, 379
// Blocks have at most 64 sub-blocks, a lane each.
constexpr float PENCIL_SECTION = 0.25f;
LEM_DEV bool pencil_box(const GridDev &G, float section, float longest, bool full)
{
    const float bound = G.mshift == 2 ? (full ? 4.0f : 8.0f) : (full ? 1.0f : 4.0f);
    return (section <= PENCIL_SECTION) & (longest <= bound) & (G.mshift >= 2) & (G.mshift <= 4);
}

// Sub-block s of block (jx, jy, jz): its first cell, and whether the beam meets it.
LEM_DEV bool pencil_sub(const GridDev &G, const BeamAxis &x, const BeamAxis &y, const BeamAxis &z,
                        int jx, int jy, int jz, int s, int &cx, int &cy, int &cz)
{
    const int b = G.mshift - 2, m = (1 << b) - 1;
    cx = (jx << G.mshift) + ((s & m) << 2);
    cy = (jy << G.mshift) + (((s >> b) & m) << 2);
    cz = (jz << G.mshift) + ((s >> (2 * b)) << 2);
    float u0 = 0.0f, u1 = 1.0f;
    const float lx = __builtin_fmaf(G.cx, (float)cx, G.lox), ly = __builtin_fmaf(G.cy, (float)cy, G.loy),
                lz = __builtin_fmaf(G.cz, (float)cz, G.loz);
    beam_clip(x, lx, __builtin_fmaf(G.cx, 4.0f, lx), u0, u1);
    beam_clip(y, ly, __builtin_fmaf(G.cy, 4.0f, ly), u0, u1);
    beam_clip(z, lz, __builtin_fmaf(G.cz, 4.0f, lz), u0, u1);
    return (u0 <= u1) & (cx < G.nx) & (cy < G.ny) & (cz < G.nz);
}

// Cell `l` of the sub-block whose first cell is (cx, cy, cz): its triangles [b, e), none
// if the beam misses its box.  up_*: the rays' direction (cells come in their order).
LEM_DEV void pencil_cell(const GridDev &G, const float4 *__restrict__ box, const BeamAxis &x,
                         const BeamAxis &y, const BeamAxis &z, int cx, int cy, int cz, int l,
                         bool up_x, bool up_y, bool up_z, int32_t &b, int32_t &e)
{
    const int ix = cx + ((l & 3) ^ (up_x ? 0 : 3)), iy = cy + (((l >> 2) & 3) ^ (up_y ? 0 : 3)),
              iz = cz + ((l >> 4) ^ (up_z ? 0 : 3));
    b = e = 0;
    if ((ix >= G.nx) | (iy >= G.ny) | (iz >= G.nz))
        return;
    const int c = (iz * G.ny + iy) * G.nx + ix;
    const float4 lo = box[2 * c], hi = box[2 * c + 1];
    float u0 = 0.0f, u1 = 1.0f;
    beam_clip(x, lo.x, hi.x, u0, u1);
    beam_clip(y, lo.y, hi.y, u0, u1);
    beam_clip(z, lo.z, hi.z, u0, u1);
    if (u0 <= u1) {
        b = __builtin_bit_cast(int32_t, lo.w);
        e = __builtin_bit_cast(int32_t, hi.w);
    }
}

// A ray's reciprocal direction and origin times it: the plane at x is t = x id + oid.
// (oid's rounding is one of the origin, the same for every plane.)
struct RaySlabs {
    float idx, idy, idz, ox, oy, oz;
};

// 1 / x to the last place or so: the hardware's estimate and one Newton step
LEM_DEV float near_recip(float x)
{
    const float y = rcpf_estimate(x);
    return __builtin_fmaf(y, __builtin_fmaf(-x, y, 1.0f), y);
}

LEM_DEV RaySlabs ray_slabs(const Ray &r)
{
    RaySlabs k;
    k.idx = near_recip(r.dx); k.idy = near_recip(r.dy); k.idz = near_recip(r.dz);
    k.ox = -r.ox * k.idx; k.oy = -r.oy * k.idy; k.oz = -r.oz * k.idz;
    return k;
}

// The t interval of the ray between the faces of a box narrows [tn, tf].
LEM_DEV void slabs_clip(const RaySlabs &k, float lx, float ly, float lz, float hx, float hy, float hz,
                        float &tn, float &tf)
{
    const float x0 = __builtin_fmaf(lx, k.idx, k.ox), x1 = __builtin_fmaf(hx, k.idx, k.ox);
    const float y0 = __builtin_fmaf(ly, k.idy, k.oy), y1 = __builtin_fmaf(hy, k.idy, k.oy);
    const float z0 = __builtin_fmaf(lz, k.idz, k.oz), z1 = __builtin_fmaf(hz, k.idz, k.oz);
    tn = fmaxf(fmaxf(tn, fminf(x0, x1)), fmaxf(fminf(y0, y1), fminf(z0, z1)));
    tf = fminf(fminf(tf, fmaxf(x0, x1)), fminf(fmaxf(y0, y1), fmaxf(z0, z1)));
}

// A ray's hits so far: dist as dda_cast keeps it; the closest hit, its triangle and
// the closest hit of another triangle.
struct RayHits {
    float dist;
    double tmin, t_next;
    int32_t id_min;
    bool hit;
};

// The cells of block (jx, jy, jz) that ray r crosses inside the block's content box,
// and their triangles (rt: the predicate's ray).  The walk begins at the box, not
// at the block: what lies before it holds no triangle of this block, and a cell
// off by one at an edge only shifts it within the eps inflation of the boxes.
template <bool ANY, int SEM>
LEM_DEV void block_walk(const Ray &r, const Ray &rt, const RaySlabs &k, const GridDev &G, uint2 qv,
                        int jx, int jy, int jz, const float4 *__restrict__ recs,
                        const float4 *__restrict__ box, RayHits &h)
{
    const float margin = 2.0f * G.eps;
    const float ox = macro_origin(G.qlx, G.cx, jx, G.mshift), oy = macro_origin(G.qly, G.cy, jy, G.mshift),
                oz = macro_origin(G.qlz, G.cz, jz, G.mshift);
    float tn = -margin, tf = h.dist + margin;
    slabs_clip(k, ox + (float)(qv.x & 255u) * G.qx, oy + (float)((qv.x >> 8) & 255u) * G.qy,
               oz + (float)((qv.x >> 16) & 255u) * G.qz, ox + (float)(qv.x >> 24) * G.qx,
               oy + (float)(qv.y & 255u) * G.qy, oz + (float)((qv.y >> 8) & 255u) * G.qz, tn, tf);
    float t_end = tf + margin;
    if (!(tn <= t_end) || (ANY && h.hit))
        return;
    const int ms = G.mshift, B = 1 << ms;
    const int lx = jx << ms, ly = jy << ms, lz = jz << ms;
    const int ux = min(lx + B, G.nx), uy = min(ly + B, G.ny), uz = min(lz + B, G.nz);
    const float te = fmaxf(tn, 0.0f);
    const int ix = clampi((int)floorf((r.ox + r.dx * te - G.lox) * G.icx), lx, ux - 1);
    const int iy = clampi((int)floorf((r.oy + r.dy * te - G.loy) * G.icy), ly, uy - 1);
    const int iz = clampi((int)floorf((r.oz + r.dz * te - G.loz) * G.icz), lz, uz - 1);
    const bool sx = r.dx > 0.0f, sy = r.dy > 0.0f, sz = r.dz > 0.0f;
    // the far face of the cell on each axis (f) and its distance; the walk ends at
    // the box or at the block's far faces, which are the same expressions
    const float Dx = G.cx * k.idx, Dy = G.cy * k.idy, Dz = G.cz * k.idz;
    const float Ex = __builtin_fmaf(G.lox, k.idx, k.ox), Ey = __builtin_fmaf(G.loy, k.idy, k.oy),
                Ez = __builtin_fmaf(G.loz, k.idz, k.oz);
    float fx = (float)(ix + (sx ? 1 : 0)), fy = (float)(iy + (sy ? 1 : 0)),
          fz = (float)(iz + (sz ? 1 : 0));
    float tx = __builtin_fmaf(fx, Dx, Ex), ty = __builtin_fmaf(fy, Dy, Ey),
          tz = __builtin_fmaf(fz, Dz, Ez);
    t_end = fminf(t_end, __builtin_fmaf((float)(sx ? ux : lx), Dx, Ex));
    t_end = fminf(t_end, __builtin_fmaf((float)(sy ? uy : ly), Dy, Ey));
    t_end = fminf(t_end, __builtin_fmaf((float)(sz ? uz : lz), Dz, Ez));
    int c = (iz * G.ny + iy) * G.nx + ix;
    for (int g = 3 * B; g > 0; --g) {
        const float4 clo = box[2 * c], chi = box[2 * c + 1];
        const int32_t b = __builtin_bit_cast(int32_t, clo.w);
        float cn = -margin, cf = h.dist + margin;
        slabs_clip(k, clo.x, clo.y, clo.z, chi.x, chi.y, chi.z, cn, cf);
        const int32_t e = cn <= cf + margin ? __builtin_bit_cast(int32_t, chi.w) : b;
        for (int32_t j = b; j < e; ++j) {
            const Tri t = load_rec(recs, j);
            if (SEM == 1) {
                if (hit_native(rt, t)) {
                    h.hit = true;
                    return;
                }
                continue;
            }
            double tt;
            if (ANY) {
                if (hit_numba(rt, rt.len, t, tt)) {
                    h.hit = true;
                    return;
                }
            } else if (hit_numba(r, r.len, t, tt)) {
                const int32_t id = rec_id(recs, j);
                if (id != h.id_min) {
                    if (tt < h.tmin) {
                        if (h.hit)
                            h.t_next = fmin(h.t_next, h.tmin);
                        h.tmin = tt;
                        h.id_min = id;
                        h.dist = (float)tt;
                        h.hit = true;
                        t_end = fminf(t_end, h.dist + margin);
                    } else if (tt < h.t_next) {
                        h.t_next = tt;
                    }
                }
            }
        }
        const float texit = fminf(tx, fminf(ty, tz));
        if (!(texit < t_end))
            break;
        // an axis whose distances are not numbers (a direction component near the
        // end of float32) is never crossed
        const bool ax = tx == texit;
        const bool ay = !ax && ty == texit;
        const bool az = !ax && !ay && tz == texit;
        if (!(ax | ay | az))
            break;
        fx += ax ? (sx ? 1.0f : -1.0f) : 0.0f;
        fy += ay ? (sy ? 1.0f : -1.0f) : 0.0f;
        fz += az ? (sz ? 1.0f : -1.0f) : 0.0f;
        const int sc = ax ? 1 : (ay ? G.nx : G.nx * G.ny);
        c += (ax ? sx : (ay ? sy : sz)) ? sc : -sc;
        tx = __builtin_fmaf(fx, Dx, Ex);
        ty = __builtin_fmaf(fy, Dy, Ey);
        tz = __builtin_fmaf(fz, Dz, Ez);
    }
}

}  // namespace lem
