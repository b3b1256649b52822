// beam_walk_host.cpp -- CPU build of the beam walk (lem_beam_walk.h): 64 rays with a
// common end, cast the way the persistent traversal casts a wavefront, checked ray by
// ray against the oracle's brute force.  Scenes and grids are those of
// grid_walk_host.cpp; the free ends are drawn in clusters of 64, from points to wide
// ones, so that beams of every width up to the refused ones occur.  Test
// infrastructure, built and run by tests/test_beam_walk_host.py.
#define main grid_walk_main
#include "grid_walk_host.cpp"
#undef main

#include "../../lyceanem-python_amd/csrc/lem_beam_walk.h"

namespace {

// One wavefront; lanes with `walk` false have no ray.  False: too wide.
template <bool ANY, int SEM>
bool beam_host(const HostGrid &H, const float *P, const std::vector<const float *> &Q, bool from_p,
               const std::vector<Ray> &r, const std::vector<Ray> &rt, const std::vector<char> &walk,
               std::vector<RayHits> &h)
{
    const GridDev &G = H.G;
    const MacroTab smq{H.qa.data(), H.qb.data(), H.axis};
    float lo[3], hi[3];
    for (int a = 0; a < 3; ++a) {
        lo[a] = hi[a] = Q[0][a];
        for (auto q : Q) {
            lo[a] = fminf(lo[a], q[a]);
            hi[a] = fmaxf(hi[a], q[a]);
        }
    }
    Beam b;
    if (!beam_of(G, P[0], P[1], P[2], lo[0], lo[1], lo[2], hi[0], hi[1], hi[2], from_p, b))
        return false;
    const size_t n = Q.size();
    std::vector<RaySlabs> k(n);
    h.resize(n);
    for (size_t i = 0; i < n; ++i) {
        k[i] = ray_slabs(r[i]);
        h[i] = RayHits{r[i].len, (double)r[i].len, __builtin_huge_val(), -1, false};
    }
    for (int s = 0; s < b.slabs; ++s) {
        const int j = b.first + b.step * s;
        int a0, na, b0, nb;
        const int cnt = beam_slab(b, j, a0, na, b0, nb);
        if (cnt > BEAM_MAX || (cnt > 0 && (na > BEAM_NA || nb > BEAM_NB)))
            return false;
        if (cnt == 0)
            continue;
        BeamAxis ax[3];
        for (int a = 0; a < 3; ++a)
            ax[a] = beam_axis(P[a], lo[a] - P[a], hi[a] - P[a], b.mrg);
        uint32_t m = beam_mask(G, smq, b.axis, ax[0], ax[1], ax[2], j, a0, na, b0, cnt);
        for (; m; m &= m - 1) {
            const int bit = __builtin_ctz(m);
            int jx, jy, jz;
            beam_block_at(b.axis, j, a0 + (bit & 7), b0 + (bit >> 3), jx, jy, jz);
            if (jx < 0 || jx >= G.mx || jy < 0 || jy >= G.my || jz < 0 || jz >= G.mz)
                std::exit(3);
            for (size_t i = 0; i < n; ++i)
                if (walk[i])
                    block_walk<ANY, SEM>(r[i], rt[i], k[i], G, smq[(jz * G.my + jy) * G.mx + jx], jx,
                                         jy, jz, H.recs.data(), H.box.data(), h[i]);
        }
    }
    if (!ANY)
        for (size_t i = 0; i < n; ++i)
            if (h[i].hit) {
                const float fs = (float)h[i].tmin;
                const double delta =
                    8.0 * (2e-7 + (double)(nextafterf(fs, __builtin_huge_valf()) - fs));
                if (h[i].t_next <= h[i].tmin + delta)
                    h[i].dist = replay_window(r[i], h[i].tmin, G, H.cell_start.data(),
                                              H.recs.data());
            }
    return true;
}

// One wavefront as a pencil, any hit; the lanes' hits.
bool pencil_host(const HostGrid &H, const float *P, const std::vector<const float *> &Q, bool from_p,
                 const std::vector<Ray> &rt, std::vector<char> &hit)
{
    const GridDev &G = H.G;
    const MacroTab smq{H.qa.data(), H.qb.data(), H.axis};
    float lo[3], hi[3];
    for (int a = 0; a < 3; ++a) {
        lo[a] = hi[a] = Q[0][a];
        for (auto q : Q) {
            lo[a] = fminf(lo[a], q[a]);
            hi[a] = fmaxf(hi[a], q[a]);
        }
    }
    Beam b;
    if (!beam_of(G, P[0], P[1], P[2], lo[0], lo[1], lo[2], hi[0], hi[1], hi[2], from_p, b))
        return false;
    BeamAxis ax[3];
    bool up[3];
    const float mrg = beam_margin(G, P[0], P[1], P[2], lo[0], lo[1], lo[2], hi[0], hi[1], hi[2]);
    for (int a = 0; a < 3; ++a) {
        ax[a] = beam_axis(P[a], lo[a] - P[a], hi[a] - P[a], mrg);
        up[a] = (lo[a] + hi[a] >= 2.0f * P[a]) == from_p;
    }
    hit.assign(Q.size(), 0);
    for (int s = 0; s < b.slabs; ++s) {
        const int j = b.first + b.step * s;
        int a0, na, b0, nb;
        const int cnt = beam_slab(b, j, a0, na, b0, nb);
        if (cnt > BEAM_MAX || (cnt > 0 && (na > BEAM_NA || nb > BEAM_NB)))
            return false;
        for (uint32_t m = cnt ? beam_mask(G, smq, b.axis, ax[0], ax[1], ax[2], j, a0, na, b0, cnt) : 0;
             m; m &= m - 1) {
            const int bit = __builtin_ctz(m);
            int jx, jy, jz;
            beam_block_at(b.axis, j, a0 + (bit & 7), b0 + (bit >> 3), jx, jy, jz);
            for (int sub = 0; sub < 1 << (3 * (G.mshift - 2)); ++sub) {
                int cx, cy, cz;
                if (!pencil_sub(G, ax[0], ax[1], ax[2], jx, jy, jz, sub, cx, cy, cz))
                    continue;
                for (int l = 0; l < 64; ++l) {
                    int32_t r0, r1;
                    pencil_cell(G, H.box.data(), ax[0], ax[1], ax[2], cx, cy, cz, l, up[0], up[1],
                                up[2], r0, r1);
                    for (int32_t r = r0; r < r1; ++r)
                        for (size_t i = 0; i < Q.size(); ++i) {
                            double tt;
                            hit[i] |= hit_numba(rt[i], rt[i].len, load_rec(H.recs.data(), r), tt);
                        }
                }
            }
        }
    }
    return true;
}

int64_t g_beams = 0, g_refused = 0;

// clusters of 64 around points of `centres`, radii of `frac` of the scene and less
std::vector<float> clusters(const std::vector<float> &centres, double size, Rng &g)
{
    std::vector<float> out;
    for (size_t c = 0; c < centres.size() / 3; ++c) {
        const double rad = c % 4 == 0 ? 0.0 : size * std::pow(10.0, g.uni(-4.0, -0.5));
        const int n = c % 7 == 6 ? 37 : 64;
        for (int i = 0; i < 64; ++i) {
            // the tail of a short cluster repeats its first point (lanes past the end)
            const size_t b = out.size() - (i < n ? 0 : 3 * i);
            if (i < n)
                push3(out, centres[3 * c] + g.uni(-rad, rad), centres[3 * c + 1] + g.uni(-rad, rad),
                      centres[3 * c + 2] + g.uni(-rad, rad));
            else
                for (int a = 0; a < 3; ++a)
                    out.push_back(out[b + a]);
        }
    }
    return out;
}

void check_beams(Scene sc, float cells_per_tri, int force_mshift, uint64_t seed)
{
    Rng g(seed);
    float lo = 1e30f, hi = -1e30f;
    for (float v : sc.tris) {
        lo = std::min(lo, v);
        hi = std::max(hi, v);
    }
    sc.src = clusters(sc.src, hi - lo, g);
    const int64_t T = (int64_t)sc.tris.size() / 9, S = (int64_t)sc.src.size() / 3,
                  K = (int64_t)sc.snk.size() / 3;
    const HostGrid H = build_grid(sc.tris, cells_per_tri, force_mshift);
    // forward: rays from the clusters to the sinks; back: the other way round
    for (int back = 0; back < 2; ++back) {
        const std::vector<float> &from = back ? sc.snk : sc.src, &to = back ? sc.src : sc.snk;
        const int64_t A = back ? K : S, B = back ? S : K;
        std::vector<uint8_t> hit(S * K), hit_n(S * K);
        std::vector<float> dist(S * K);
        orc_visibility_dense(from.data(), A, to.data(), B, sc.tris.data(), T, 0, 0, 0, hit.data(),
                             dist.data(), 0);
        orc_visibility_dense(from.data(), A, to.data(), B, sc.tris.data(), T, 1, 1, 0,
                             hit_n.data(), nullptr, 0);
        int64_t bad = 0, rays = 0, refused = 0, beams = 0;
        for (int64_t k = 0; k < K; ++k)
            for (int64_t s0 = 0; s0 < S; s0 += 64)
                for (int mode = 0; mode < 5; ++mode) {
                    // closest, any, any walked from the other end, native, native walked so
                    const bool rev = mode == 2 || mode == 4;
                    const bool from_p = (back != 0) != rev;  // P: the sink
                    std::vector<const float *> Q;
                    std::vector<Ray> r, rt;
                    std::vector<char> walk;
                    for (int i = 0; i < 64; ++i) {
                        const float *q = &sc.src[3 * (s0 + i)], *p = &sc.snk[3 * k];
                        const float *a = back ? p : q, *b = back ? q : p;
                        Q.push_back(q);
                        rt.push_back(charge(a[0], a[1], a[2], b[0], b[1], b[2]));
                        r.push_back(rev ? charge(b[0], b[1], b[2], a[0], a[1], a[2]) : rt.back());
                        const Ray &w = r.back();
                        walk.push_back(w.len > 0.0f && w.dx != 0.0f && w.dy != 0.0f &&
                                       w.dz != 0.0f && std::isfinite(w.len));
                    }
                    std::vector<RayHits> h;
                    const float *P = &sc.snk[3 * k];
                    const bool ok =
                        mode == 0   ? beam_host<false, 0>(H, P, Q, from_p, r, rt, walk, h)
                        : mode <= 2 ? beam_host<true, 0>(H, P, Q, from_p, r, rt, walk, h)
                                    : beam_host<true, 1>(H, P, Q, from_p, r, rt, walk, h);
                    ++beams;
                    if (mode == 0)  // the same rays one by one, blocks skipped in a loop of their own
                        for (int i = 0; i < 64; ++i)
                            if (walk[i]) {
                                const int64_t at = back ? k * S + s0 + i : (s0 + i) * K + k;
                                float d = r[i].len;
                                const bool hc = closest_cast(
                                    r[i], d, H.G, H.cell_start.data(), H.recs.data(), H.box.data(),
                                    MacroTab{H.qa.data(), H.qb.data(), H.axis});
                                bad += hc != hit[at] || std::memcmp(&d, &dist[at], 4) != 0;
                            }
                    if ((mode == 1 || mode == 2) && H.info.mshift >= 2 && H.info.mshift <= 4) {
                        std::vector<char> p;
                        if (pencil_host(H, P, Q, from_p, rt, p) != ok)
                            ++bad;
                        for (int i = 0; ok && i < 64; ++i)
                            bad += p[i] != hit[back ? k * S + s0 + i : (s0 + i) * K + k];
                    }
                    if (!ok) {
                        ++refused;
                        continue;
                    }
                    for (int i = 0; i < 64; ++i)
                        if (walk[i]) {
                            const int64_t at = back ? k * S + s0 + i : (s0 + i) * K + k;
                            ++rays;
                            bad += h[i].hit != (mode >= 3 ? hit_n[at] : hit[at]);
                            bad += mode == 0 && std::memcmp(&h[i].dist, &dist[at], 4) != 0;
                        }
                }
        g_bad += bad;
        g_rays += rays;
        g_beams += beams;
        g_refused += refused;
        std::printf("%-14s cells/tri %.0f mshift %d back %d: %lld beams, %lld refused, %lld rays, "
                    "%lld mismatches\n",
                    sc.name.c_str(), cells_per_tri, H.info.mshift, back, (long long)beams,
                    (long long)refused, (long long)rays, (long long)bad);
    }
}

}  // namespace

int main(int argc, char **argv)
{
    const bool quick = argc > 1;
    const int f = quick ? 1 : 2;
    std::vector<Scene> scenes = {terrain(1, 24, 18, 8 * f, 9 * f), terrain(2, 60, 40, 8 * f, 9 * f),
                                 terrain_sky(3, 40, 30, 8 * f, 9 * f),
                                 cell_boundaries(terrain(4, 30, 20, 0, 0), 2.0f, 5, 8 * f, 9 * f),
                                 clutter(6, 300, 8 * f, 9 * f, 0.4),
                                 clutter(7, 4000, 8 * f, 9 * f, 0.1), planes(8, 500, 9 * f, 9 * f),
                                 far_scene(9, 800, 8 * f, 9 * f)};
    for (const Scene &sc : scenes)
        for (float cells : {1.0f, 2.0f, 4.0f})
            for (int ms : {-1, 0, 1, 3})
                if (cells == 2.0f ? !quick || ms <= 0 : !quick && ms == -1)
                    check_beams(sc, cells, ms, 11);
    std::printf("total: %lld rays of %lld beams, %lld refused, %lld mismatches\n",
                (long long)g_rays, (long long)g_beams, (long long)g_refused, (long long)g_bad);
    return g_bad != 0;
}
