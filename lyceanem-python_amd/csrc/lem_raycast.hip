// lem_raycast.hip -- brute-force Moller-Trumbore visibility for gfx950.
//
// Replaces kernel1Dv3 (rayfunctions.py:212-244) as launched by
// launchRaycaster1Dv3 / chunkingRaycaster1Dv3 (rayfunctions.py:1951-2017,
// 2102-2369), and the native raycast_brute_force (raycasting_brute_force.cuh:68-88).
//
// Layout: one thread per ray, 256 (or 512) rays per block.  The block streams the
// triangle table through LDS in tiles of 256 (v0, e1, e2 padded to 48 B so a
// wave reads a triangle with three broadcast ds_read_b128).  Every ray meets the
// triangles in table order, so the closest-hit mode reproduces kernel1Dv3's
// shrinking window exactly.  The any-hit mode stops a ray at its first accepted
// hit and stops the block as soon as all its rays are done.  The dense kernel,
// whose blocks share one origin, first drops what cannot be hit from there; the
// explicit list tests every triangle.
#include "lem_device.h"
#include "lem_internal.h"
#include "lem_shared_origin.h"
#include "../../include/lem.h"

namespace lem {

constexpr int RC_BLOCK = 256;
constexpr int RC_TILE = 256;
// k_visibility_dense: workgroups of 512 rays from this many sinks up, of 256
// below.  Rays are sorted by direction within a workgroup, so larger ones make
// tighter groups; small launches need the workgroups (16,471 sinks, 2,000
// triangles, closest hit: 6.3 ms with 512, 9.6 with 256; 703 sinks: 225 and 204 us).
constexpr int64_t DENSE_WIDE_SINKS = 4096;
// ... and sorted from this many triangles up (60 triangles: 75 us unsorted, 95 sorted)
constexpr int64_t DENSE_SORT_TRIS = 128;

struct alignas(16) TriLds {
    float v0x, v0y, v0z, e1x;
    float e1y, e1z, e2x, e2y;
    float e2z, pad0, pad1, pad2;
};

__device__ __forceinline__ void stage_tile(TriLds *s_tri, const float *__restrict__ tris,
                                           int64_t base, int64_t T)
{
    int64_t j = base + threadIdx.x;
    TriLds L;
    if (j < T) {
        Tri t = make_tri(tris + 9 * j);
        L.v0x = t.v0x; L.v0y = t.v0y; L.v0z = t.v0z;
        L.e1x = t.e1x; L.e1y = t.e1y; L.e1z = t.e1z;
        L.e2x = t.e2x; L.e2y = t.e2y; L.e2z = t.e2z;
    } else {
        L.v0x = L.v0y = L.v0z = 0.0f;
        L.e1x = L.e1y = L.e1z = 0.0f;
        L.e2x = L.e2y = L.e2z = 0.0f;
    }
    L.pad0 = L.pad1 = L.pad2 = 0.0f;
    s_tri[threadIdx.x] = L;
}

__device__ __forceinline__ Tri load_tri(const TriLds *s_tri, int j)
{
    TriLds L = s_tri[j];
    Tri t;
    t.v0x = L.v0x; t.v0y = L.v0y; t.v0z = L.v0z;
    t.e1x = L.e1x; t.e1y = L.e1y; t.e1z = L.e1z;
    t.e2x = L.e2x; t.e2y = L.e2y; t.e2z = L.e2z;
    return t;
}

// Walk every triangle (or until the first hit with ANY) for one ray.
// SEM 0 = numba predicate + kernel1Dv3 dist update, SEM 1 = native culled.
template <int SEM, bool ANY>
__device__ __forceinline__ void tile_walk(const TriLds *s_tri, int n, const Ray &r,
                                          float &dist, bool &hit)
{
    for (int j = 0; j < n; ++j) {
        Tri t = load_tri(s_tri, j);
        if (SEM == 0) {
            // hit_numba accepts t < dist - 2e-7 only, so an accepted hit is
            // always closer than dist (kernel1Dv3's t < ray.dist test)
            double tt;
            if (hit_numba(r, dist, t, tt)) {
                dist = (float)tt;
                hit = true;
                if (ANY)
                    return;
            }
        } else {
            if (hit_native(r, t)) {
                hit = true;
                if (ANY)
                    return;
            }
        }
    }
}

// 21-bit Morton key of a unit direction (7 bits an axis).
__device__ __forceinline__ uint32_t direction_key(float dx, float dy, float dz)
{
    uint32_t key = 0;
    const float d[3] = {dx, dy, dz};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const float f = d[a] * 63.5f + 64.0f;
        uint32_t q = f > 0.0f ? (f < 127.0f ? (uint32_t)f : 127u) : 0u;  // NaN -> 0
        q = (q | (q << 8)) & 0x0000f00fu;
        q = (q | (q << 4)) & 0x000c30c3u;
        q = (q | (q << 2)) & 0x00249249u;
        key |= q << a;
    }
    return key;
}

// Sorts N (a power of two, the block's threads) distinct keys in LDS (bitonic).
template <int N>
__device__ __forceinline__ void sort_keys(uint32_t *s)
{
    for (int size = 2; size <= N; size <<= 1)
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            __syncthreads();
            const int p = threadIdx.x;
            if (p < N / 2) {
                const int lo = 2 * p - (p & (stride - 1)), hi = lo + stride;
                const uint32_t a = s[lo], b = s[hi];
                const bool up = (lo & size) == 0;
                if ((a > b) == up) {
                    s[lo] = b;
                    s[hi] = a;
                }
            }
        }
}

// Centre and half width of one component over the wave's lanes (those with
// `skip` left out), widened by their own rounding; uniform over the wave.  0 and 0
// when all are left out or are NaN (a zero-length ray hits nothing).
__device__ __forceinline__ void axis_box(float d, bool skip, float &c, float &h)
{
    float lo = skip ? 2.0f : d, hi = skip ? -2.0f : d;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        lo = fminf(lo, __shfl_xor(lo, off));
        hi = fmaxf(hi, __shfl_xor(hi, off));
    }
    const bool some = lo <= hi;
    c = some ? 0.5f * (lo + hi) : 0.0f;
    h = some ? 0.5f * (hi - lo) + 1e-6f : 0.0f;
}

// Dense S x K: block b owns source s = b / nbk and the BLK sinks from
// (b % nbk) * BLK.  hit_bits is S x W64 words; bit (k % 64) of word (k / 64) set =
// ray blocked.
//
// All rays of a block share their origin, so a triangle is tested by the linear
// tests of lem_shared_origin.h (16 operations a ray instead of the predicate's
// about 57) and the predicate itself runs, as written and in table order, only
// on what they leave.
// The block's rays are sorted by direction, 64 neighbours to a wave, and a wave
// first drops, a lane a triangle, the triangles that no direction in its box can
// hit: by the same three tests over the box, and by the ball of directions the
// triangle fills (shared_origin_tests).  A lane keeps the last triangle its ray
// might hit (`pend`); the predicate runs when one of the wave's lanes finds its
// next, for all that hold one -- rays meet their few candidates at different
// triangles, so one at a time the predicate would run with a lane or two.
//
// Bound: VALU issue, and LDS reads of the triangles a wave keeps.  Before, every
// ray ran the predicate on every triangle.  32 x 32 sources, 16,471 sinks, 2,000
// triangles of metre size half a metre away: closest hit 29.0 -> 5.8 ms, any hit
// 20.0 -> 4.3; 16 x 16 on a cylinder of 5,488 triangles, 7,381 sinks: any hit 7.3
// -> 1.05 ms.  (Measured and left: the linear tests alone, 10.5 and 4.7 ms; four
// rays a lane for fewer LDS reads, 7.4 and 4.6; waves that load and prepare
// triangles by themselves, without LDS, 8.9 and 2.3.)
template <int SEM, bool ANY, int BLK, int NT>
__global__ __launch_bounds__(BLK) void k_visibility_dense(
    const float *__restrict__ src, const float *__restrict__ snk, int64_t K,
    const float *__restrict__ tris, int64_t T, int skip_self,
    unsigned long long *__restrict__ hit_bits, int64_t W64, float *__restrict__ dist_out,
    int64_t nbk)
{
    __shared__ uint32_t s_key[BLK];
    __shared__ unsigned long long s_bits[BLK / 64];
    // a tile of triangles: as the predicate reads them, their linear tests and
    // balls (one entry more: never hit)
    __shared__ TriLds s_tri[RC_TILE];
    __shared__ float4 s_a[RC_TILE + 1], s_u[RC_TILE + 1], s_v[RC_TILE + 1], s_ball[RC_TILE];
    const int64_t s = (int64_t)blockIdx.x / nbk;
    const int64_t k0 = ((int64_t)blockIdx.x % nbk) * BLK;
    const float ox = src[3 * s], oy = src[3 * s + 1], oz = src[3 * s + 2];
    const int lane = threadIdx.x & 63;
    {
        // which ray a lane takes: the block's rays in a Morton order of their
        // directions
        const int64_t k = k0 + threadIdx.x;
        uint32_t key = threadIdx.x | 0xfffffe00u;
        if (k < K && T >= DENSE_SORT_TRIS) {
            const Ray r = charge(ox, oy, oz, snk[3 * k], snk[3 * k + 1], snk[3 * k + 2]);
            key = threadIdx.x | direction_key(r.dx, r.dy, r.dz) << 9;
        }
        s_key[threadIdx.x] = key;
        if (threadIdx.x < BLK / 64)
            s_bits[threadIdx.x] = 0ull;
        if (threadIdx.x < 3)
            (threadIdx.x == 0 ? s_a : threadIdx.x == 1 ? s_u : s_v)[RC_TILE] =
                make_float4(0.0f, 0.0f, 0.0f, -__builtin_huge_valf());
        if (T >= DENSE_SORT_TRIS)
            sort_keys<BLK>(s_key);
        __syncthreads();
    }
    const int loc = s_key[threadIdx.x] & 511u;
    const int64_t k = k0 + loc;
    const bool active = k < K;
    const int64_t kk = active ? k : 0;
    const Ray r = charge(ox, oy, oz, snk[3 * kk], snk[3 * kk + 1], snk[3 * kk + 2]);
    float dist = r.len;
    int pend = -1;
    bool hit = false, done = !active || (skip_self && s == k);
    // box of the group's directions
    float bcx, bcy, bcz, bhx, bhy, bhz;
    axis_box(r.dx, done, bcx, bhx);
    axis_box(r.dy, done, bcy, bhy);
    axis_box(r.dz, done, bcz, bhz);
    // the predicate on the lanes' pending triangles
    auto resolve = [&]() {
        if (pend >= 0) {
            const Tri t = load_tri(s_tri, pend);
            if (SEM == 0) {
                // hit_numba accepts t < dist - 2e-7 only, so an accepted hit is
                // always closer than dist (kernel1Dv3's t < ray.dist test)
                double tt;
                if (hit_numba(r, dist, t, tt)) {
                    dist = (float)tt;
                    hit = true;
                }
            } else if (hit_native(r, t)) {
                hit = true;
            }
            if (ANY)
                done = done || hit;
            pend = -1;
        }
    };
    for (int64_t base = 0; base < T; base += RC_TILE) {
        __syncthreads();
        if (threadIdx.x < RC_TILE) {
            stage_tile(s_tri, tris, base, T);
            float4 a = make_float4(0.0f, 0.0f, 0.0f, -__builtin_huge_valf()), u = a, v = a;
            float4 ball = make_float4(0.0f, 0.0f, 0.0f, 4.0f);
            if (base + threadIdx.x < T)
                shared_origin_tests<SEM>(load_tri(s_tri, threadIdx.x), ox, oy, oz, a, u, v, ball);
            s_a[threadIdx.x] = a;
            s_u[threadIdx.x] = u;
            s_v[threadIdx.x] = v;
            s_ball[threadIdx.x] = ball;
        }
        __syncthreads();
        const int n = (int)((T - base) < RC_TILE ? (T - base) : RC_TILE);
        for (int j0 = 0; j0 < n; j0 += 64) {
            // which of the next 64 triangles the group can hit, a lane a triangle
            unsigned long long live;
            {
                const float4 a = s_a[j0 + lane], u = s_u[j0 + lane], v = s_v[j0 + lane];
                const float4 ball = s_ball[j0 + lane];
                live = __ballot(!shared_origin_box_out(a, u, v, ball, bcx, bcy, bcz, bhx, bhy, bhz));
            }
            if (__ballot(!done) == 0ull)
                break;
            while (live) {
                // NT triangles at a time, so that their LDS reads and dot
                // products overlap; past the last one the entry never hit
                int jj[NT];
                float4 a[NT], u[NT], v[NT];
#pragma unroll
                for (int q = 0; q < NT; ++q) {
                    jj[q] = live ? j0 + __builtin_ctzll(live) : RC_TILE;
                    live &= live - 1;
                    a[q] = s_a[jj[q]];
                    u[q] = s_u[jj[q]];
                    v[q] = s_v[jj[q]];
                }
#pragma unroll
                for (int q = 0; q < NT; ++q) {
                    const bool out = shared_origin_out(r, dist, a[q], u[q], v[q]);
                    const bool cand = !out & !done;
                    if (__ballot(cand)) {
                        if (__ballot(cand & (pend >= 0)))
                            resolve();
                        if (cand)
                            pend = jj[q];
                    }
                }
            }
        }
        resolve();
        if (ANY) {
            if (__syncthreads_and(done ? 1 : 0))
                break;
        }
    }
    if (hit)
        atomicOr(&s_bits[loc >> 6], 1ull << (loc & 63));
    if (dist_out && active)
        dist_out[s * K + k] = dist;
    __syncthreads();
    if (threadIdx.x < BLK / 64) {
        const int64_t word = (k0 >> 6) + threadIdx.x;
        if (word < W64)
            hit_bits[s * W64 + word] = s_bits[threadIdx.x];
    }
}

// Explicit rays: pair i = (origin point, target point), 0-based rows of the
// unified N x 3 point table.  Outputs kernel1Dv3's `intersect` and `dist`.
template <int SEM, bool ANY>
__global__ __launch_bounds__(RC_BLOCK) void k_raycast_pairs(
    const float *__restrict__ pts, int64_t N, const int32_t *__restrict__ pairs, int64_t R,
    const float *__restrict__ tris, int64_t T, uint8_t *__restrict__ intersect,
    float *__restrict__ dist_out)
{
    __shared__ TriLds s_tri[RC_TILE];
    const int64_t i = (int64_t)blockIdx.x * RC_BLOCK + threadIdx.x;
    const bool active = i < R;
    Ray r;
    float dist = 0.0f;
    bool hit = false;
    bool done = !active;
    bool bad = false;
    {
        int64_t ii = active ? i : 0;
        int64_t a = pairs[2 * ii], b = pairs[2 * ii + 1];
        // Rows outside the point table are reported (intersect = 0xFF), never read.
        if (a < 0 || a >= N || b < 0 || b >= N) {
            bad = true;
            a = 0;
            b = 0;
            done = true;
        }
        r = charge(pts[3 * a], pts[3 * a + 1], pts[3 * a + 2], pts[3 * b], pts[3 * b + 1],
                   pts[3 * b + 2]);
        dist = r.len;
    }
    for (int64_t base = 0; base < T; base += RC_TILE) {
        __syncthreads();
        stage_tile(s_tri, tris, base, T);
        __syncthreads();
        int n = (int)((T - base) < RC_TILE ? (T - base) : RC_TILE);
        if (!done) {
            tile_walk<SEM, ANY>(s_tri, n, r, dist, hit);
            if (ANY && hit)
                done = true;
        }
        if (ANY) {
            if (__syncthreads_and(done ? 1 : 0))
                break;
        }
    }
    if (active) {
        intersect[i] = bad ? 0xFF : (hit ? 1 : 0);
        if (dist_out)
            dist_out[i] = dist;
    }
}

}  // namespace lem

using namespace lem;

extern "C" int lem_visibility_dense(const float *src, int64_t S, const float *snk, int64_t K,
                                    const float *tris, int64_t T, int semantics, int flags,
                                    uint64_t *hit_bits, float *dist, void *stream)
{
    clear_error();
    LEM_REQUIRE(S >= 0 && K >= 0 && T >= 0, "lem_visibility_dense: negative size");
    LEM_REQUIRE(semantics == LEM_SEM_NUMBA || semantics == LEM_SEM_NATIVE,
                "lem_visibility_dense: unknown semantics");
    if (S == 0 || K == 0)
        return OK;
    LEM_REQUIRE(src && snk && hit_bits, "lem_visibility_dense: null pointer");
    LEM_REQUIRE(T == 0 || tris, "lem_visibility_dense: null triangle table");
    const bool any = (flags & LEM_VIS_ANY_HIT) != 0;
    const int skip_self = (flags & LEM_VIS_SKIP_SELF) ? 1 : 0;
    LEM_REQUIRE(!(any && dist && semantics == LEM_SEM_NUMBA),
                "lem_visibility_dense: dist needs the closest-hit mode (no LEM_VIS_ANY_HIT)");
    const int64_t W64 = ceil_div(K, 64);
    const bool wide = K >= DENSE_WIDE_SINKS;
    const int64_t nbk = ceil_div(K, wide ? 512 : 256);
    LEM_REQUIRE(S * ceil_div(K, RC_BLOCK) <= 2147483647LL,
                "lem_visibility_dense: S*K too large for one launch");
    dim3 grid((unsigned)(S * nbk));
    hipStream_t st = as_stream(stream);
    unsigned long long *hb = reinterpret_cast<unsigned long long *>(hit_bits);
#define LEM_DENSE(SEM, ANY)                                                                   \
    do {                                                                                      \
        if (wide)                                                                             \
            hipLaunchKernelGGL((k_visibility_dense<SEM, ANY, 512, 2>), grid, dim3(512), 0, st, \
                               src, snk, K, tris, T, skip_self, hb, W64, dist, nbk);          \
        else                                                                                  \
            hipLaunchKernelGGL((k_visibility_dense<SEM, ANY, 256, 4>), grid, dim3(256), 0, st, \
                               src, snk, K, tris, T, skip_self, hb, W64, dist, nbk);          \
    } while (0)
    if (semantics == LEM_SEM_NATIVE)
        LEM_DENSE(1, true);
    else if (any)
        LEM_DENSE(0, true);
    else
        LEM_DENSE(0, false);
#undef LEM_DENSE
    return check_launch("k_visibility_dense");
}

extern "C" int lem_raycast_pairs(const float *points, int64_t n_points, const int32_t *pairs,
                                 int64_t n_rays, const float *tris, int64_t T, int semantics,
                                 int flags, uint8_t *intersect, float *dist, void *stream)
{
    clear_error();
    LEM_REQUIRE(n_points >= 0 && n_rays >= 0 && T >= 0, "lem_raycast_pairs: negative size");
    LEM_REQUIRE(semantics == LEM_SEM_NUMBA || semantics == LEM_SEM_NATIVE,
                "lem_raycast_pairs: unknown semantics");
    if (n_rays == 0)
        return OK;
    LEM_REQUIRE(points && pairs && intersect, "lem_raycast_pairs: null pointer");
    LEM_REQUIRE(n_points > 0, "lem_raycast_pairs: empty point table");
    LEM_REQUIRE(T == 0 || tris, "lem_raycast_pairs: null triangle table");
    const bool any = (flags & LEM_VIS_ANY_HIT) != 0;
    LEM_REQUIRE(!(any && dist && semantics == LEM_SEM_NUMBA),
                "lem_raycast_pairs: dist needs the closest-hit mode (no LEM_VIS_ANY_HIT)");
    LEM_REQUIRE(ceil_div(n_rays, RC_BLOCK) <= 2147483647LL, "lem_raycast_pairs: too many rays");
    dim3 grid((unsigned)ceil_div(n_rays, RC_BLOCK));
    hipStream_t st = as_stream(stream);
    if (semantics == LEM_SEM_NUMBA) {
        if (any)
            hipLaunchKernelGGL((k_raycast_pairs<0, true>), grid, dim3(RC_BLOCK), 0, st, points,
                               n_points, pairs, n_rays, tris, T, intersect, dist);
        else
            hipLaunchKernelGGL((k_raycast_pairs<0, false>), grid, dim3(RC_BLOCK), 0, st, points,
                               n_points, pairs, n_rays, tris, T, intersect, dist);
    } else {
        hipLaunchKernelGGL((k_raycast_pairs<1, true>), grid, dim3(RC_BLOCK), 0, st, points, n_points,
                           pairs, n_rays, tris, T, intersect, dist);
    }
    return check_launch("k_raycast_pairs");
}
