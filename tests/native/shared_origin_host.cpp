// shared_origin_host.cpp -- CPU check of the linear tests of
// lyceanem-python_amd/csrc/lem_shared_origin.h: no triangle that the predicate
// accepts (hit_numba, hit_native, evaluated as written) may be dropped, neither
// for the ray itself nor for a box of directions around it.  Test
// infrastructure, built and run by tests/test_shared_origin_host.py.
//
// Triangles from 1 mm to 100 m, origins from inside their plane to 1e5 sizes
// away, and directions at their vertices, edges and insides, along their plane,
// and anywhere, each with rounding-sized and larger offsets: what is accepted by
// rounding alone (an origin within a rounding error of the plane) is included.
#include "lem_host_shim.h"

#include "../../lyceanem-python_amd/csrc/lem_shared_origin.h"

#include <cstdio>

using namespace lem;

namespace {
struct Rng {
    uint64_t s;
    uint64_t next()
    {
        uint64_t z = (s += 0x9e3779b97f4a7c15ull);
        z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
        z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
        return z ^ (z >> 31);
    }
    double uni(double a, double b) { return a + (b - a) * (double)(next() >> 11) * 0x1.0p-53; }
    double mag(double lo, double hi) { return std::exp(uni(std::log(lo), std::log(hi))); }
    double sgn() { return (next() & 1) ? 1.0 : -1.0; }
    int pick(int n) { return (int)(next() % (uint64_t)n); }
};
}  // namespace

int main()
{
    Rng g{12345};
    long accepted = 0, spurious = 0, native = 0, lost = 0, lost_box = 0, kept = 0, tests = 0;
    for (int it = 0; it < 600000; ++it) {
        const double size = g.mag(1e-3, 1e2);
        float t9[9];
        const double off = g.pick(3) ? 0.0 : g.mag(1e-2, 1e3);
        for (int i = 0; i < 9; ++i)
            t9[i] = (float)(off * (1 + i % 3) + size * g.uni(-1, 1));
        if (g.pick(8) == 0)  // sliver
            for (int a = 0; a < 3; ++a)
                t9[6 + a] = (float)(t9[3 + a] + (t9[a] - t9[3 + a]) * 0.3 + size * 1e-5 * g.uni(-1, 1));
        const Tri T = make_tri(t9);
        // a point of the plane (barycentric, often an edge or vertex)
        auto bary = [&](double out[3], bool inside) {
            double u = g.uni(0, 1), v = g.uni(0, 1 - u);
            if (!inside) {
                u = g.uni(-3, 3);
                v = g.uni(-3, 3);
            } else if (g.pick(3) == 0) {
                u = g.pick(2);
                v = u ? 0 : g.pick(2);
            } else if (g.pick(3) == 0) {
                u = 0;
            }
            const double e1[3] = {T.e1x, T.e1y, T.e1z}, e2[3] = {T.e2x, T.e2y, T.e2z};
            for (int a = 0; a < 3; ++a)
                out[a] = t9[a] + u * e1[a] + v * e2[a];
        };
        double n[3] = {(double)T.e1y * T.e2z - (double)T.e1z * T.e2y,
                       (double)T.e1z * T.e2x - (double)T.e1x * T.e2z,
                       (double)T.e1x * T.e2y - (double)T.e1y * T.e2x};
        const double nn = std::sqrt(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]) + 1e-300;
        double o[3];
        const int kind = g.pick(4);
        bary(o, g.pick(3) == 0);
        const double h = kind == 0 ? 0.0 : kind == 1 ? size * g.mag(1e-9, 1e-3) : size * g.mag(1e-3, 1e5);
        for (int a = 0; a < 3; ++a)
            o[a] += g.sgn() * h * n[a] / nn + (kind == 3 ? size * g.mag(1e-2, 1e5) * g.uni(-1, 1) : 0.0);
        const float ox = (float)o[0], oy = (float)o[1], oz = (float)o[2];
        const float4 none = make_float4(0, 0, 0, -__builtin_huge_valf());
        float4 a0 = none, u0 = none, v0 = none, b0 = make_float4(0, 0, 0, 4);
        float4 a1 = none, u1 = none, v1 = none, b1 = make_float4(0, 0, 0, 4);
        shared_origin_tests<0>(T, ox, oy, oz, a0, u0, v0, b0);
        shared_origin_tests<1>(T, ox, oy, oz, a1, u1, v1, b1);
        for (int q = 0; q < 8; ++q) {
            double p[3];
            bary(p, g.pick(3) != 0);
            const double far = g.pick(2) ? 1.0 + g.mag(1e-6, 1e4) : 1.0;
            const double noise = g.pick(2) ? size * g.mag(1e-9, 1e-1) : 0.0;
            float k[3];
            for (int a = 0; a < 3; ++a)
                k[a] = (float)(o[a] + (p[a] - o[a]) * far * (g.pick(16) ? 1 : -1) + noise * g.uni(-1, 1));
            if (g.pick(6) == 0) {  // along the plane, any way
                double e[3] = {g.uni(-1, 1), g.uni(-1, 1), g.uni(-1, 1)};
                const double d = (e[0] * n[0] + e[1] * n[1] + e[2] * n[2]) / (nn * nn);
                const double L = size * g.mag(1e-1, 1e4);
                for (int a = 0; a < 3; ++a)
                    k[a] = (float)(o[a] + L * (e[a] - d * n[a] * (1 - g.sgn() * g.mag(1e-8, 1e-4))));
            }
            const Ray r = charge(ox, oy, oz, k[0], k[1], k[2]);
            ++tests;
            double tt = 0.0;
            const bool hn = hit_numba(r, r.len, T, tt), hv = hit_native(r, T);
            const bool out = shared_origin_out(r, r.len, a0, u0, v0);
            kept += !out;
            const double w = g.mag(1e-6, 1.0);
            const float cx = (float)(r.dx + w * g.uni(-1, 1)), cy = (float)(r.dy + w * g.uni(-1, 1)),
                        cz = (float)(r.dz + w * g.uni(-1, 1));
            const float hx = std::fabs(r.dx - cx) + 1e-6f, hy = std::fabs(r.dy - cy) + 1e-6f,
                        hz = std::fabs(r.dz - cz) + 1e-6f;
            if (hn) {
                ++accepted;
                lost += out || shared_origin_out(r, (float)(tt * (1 + 1e-6) + 1e-6), a0, u0, v0);
                lost_box += shared_origin_box_out(a0, u0, v0, b0, cx, cy, cz, hx, hy, hz);
                // does the point hit lie far outside the triangle's own extent?
                const double c[3] = {t9[0] + (T.e1x + T.e2x) / 3, t9[1] + (T.e1y + T.e2y) / 3,
                                     t9[2] + (T.e1z + T.e2z) / 3};
                double far2 = 0;
                const double d[3] = {r.dx, r.dy, r.dz}, oo[3] = {ox, oy, oz};
                for (int a = 0; a < 3; ++a)
                    far2 += (oo[a] + tt * d[a] - c[a]) * (oo[a] + tt * d[a] - c[a]);
                spurious += far2 > 25 * size * size;
            }
            if (hv) {
                ++native;
                lost += shared_origin_out(r, r.len, a1, u1, v1);
                lost_box += shared_origin_box_out(a1, u1, v1, b1, cx, cy, cz, hx, hy, hz);
            }
        }
    }
    std::printf("%ld rays: %ld accepted (numba; %ld far from the triangle), %ld native, %ld kept, "
                "%ld lost, %ld lost by box\n", tests, accepted, spurious, native, kept, lost, lost_box);
    return lost || lost_box ? 1 : 0;
}
