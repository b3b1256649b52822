// lem_time.hip -- time-domain propagation of ray paths (gfx950).
//
// Replaces timedomainkernal (empropagation.py:1345-1612) behind TimeDomainv3
// (empropagation.py:2910-3170) and models/time_domain.py:
//   k_time_paths : per path row, the real polarisation vector carried along the
//                  path (projections and point weights, timedomainkernal's
//                  ray_component), scaled by |product of lossy_propagation
//                  factors|, and the arrival time (path length / c + the
//                  imaginary parts of the point weights, the reference's delay
//                  convention).  float64, with the float32 roundings the
//                  reference applies inside lossy_propagation.
//   k_time_wake  : wake time = min(1 s, earliest arrival) -- the reference's
//                  atomic minimum from an initial 1 s, taken over all paths
//                  before any path is placed (the reference reads it after a
//                  block-level barrier only, so its value is launch-order
//                  dependent).
//   k_time_map   : the excitation placed at each path's start sample
//                  floor((arrival - wake) / (1 / fs)) (Python's float floor
//                  division), summed per (source, sink) slot in path order --
//                  no atomics, deterministic.  out[slot][n][c] float64.
//   trace        : the same summed over every path (the source and sink sums
//                  of time_domain.calculate_scattering), out[n][c]: the paths'
//                  amplitudes summed per start sample in a fixed order, then
//                  the excitation convolution -- O(V + N E) instead of the
//                  reference's V x E atomic additions, and deterministic.
#include "lem_device.h"
#include "lem_internal.h"
#include "../../include/lem.h"

#include <math.h>

#include <algorithm>

#include <hipcub/hipcub.hpp>

namespace lem {

constexpr int TB = 256;
constexpr double LIGHT_SPEED = 299792458.0;  // scipy.constants.c

// point i of the table, with the reference's negative-index wrap (a zero
// entry of the 1-based index reads point -1, the last one)
LEM_DEV int64_t wrap_point(int32_t one_based, int64_t N)
{
    int64_t i = (int64_t)one_based - 1;
    return i < 0 ? i + N : i;
}

// calc_sep (empropagation.py:82-93): float64 length of float32 differences
LEM_DEV double sep64(const float *__restrict__ pos, int64_t a, int64_t b)
{
    const double dx = (double)(pos[3 * b] - pos[3 * a]);
    const double dy = (double)(pos[3 * b + 1] - pos[3 * a + 1]);
    const double dz = (double)(pos[3 * b + 2] - pos[3 * a + 2]);
    return sqrt(dx * dx + dy * dy + dz * dz);
}

// |lossy_propagation(a -> b)| (empropagation.py:768-801): length rounded to
// float32, float32 direction and obliquity dot product, 1/length rounded to
// float32 inside dG; magnitude of
//   -(1/2pi) (-(alpha + j beta) - 1/len) e^{-(alpha + j beta) len} / len (d.n_b).
LEM_DEV double loss_mag(const float *__restrict__ pos, const float *__restrict__ nrm, int64_t a,
                        int64_t b, double alpha, double beta)
{
    const float dx = pos[3 * b] - pos[3 * a], dy = pos[3 * b + 1] - pos[3 * a + 1],
                dz = pos[3 * b + 2] - pos[3 * a + 2];
    const double norm = sqrt((double)dx * dx + (double)dy * dy + (double)dz * dz);
    const float len = (float)norm;
    const float ux = (float)((double)dx / norm), uy = (float)((double)dy / norm),
                uz = (float)((double)dz / norm);
    float dot = ux * nrm[3 * b] + uy * nrm[3 * b + 1];
    dot = dot + uz * nrm[3 * b + 2];
    const double inv = 1.0 / (double)len;
    const double inv32 = (double)(float)inv;
    const double re = alpha + inv32, im = beta;
    // lossless: e^{-0 len} = 1 without evaluating the exponential
    const double att = alpha != 0.0 ? exp(-alpha * (double)len) : 1.0;
    return (1.0 / (2.0 * M_PI)) * sqrt(re * re + im * im) * att * inv * fabs((double)dot);
}

// (I - d d^T) v for the unit float64 direction a -> b (calc_dv into a float64
// array, then sourcelaunchtransformGPU's u/v projection)
LEM_DEV void project_dir(const float *__restrict__ pos, int64_t a, int64_t b, double v[3])
{
    const double dx = (double)(pos[3 * b] - pos[3 * a]);
    const double dy = (double)(pos[3 * b + 1] - pos[3 * a + 1]);
    const double dz = (double)(pos[3 * b + 2] - pos[3 * a + 2]);
    const double in = 1.0 / sqrt(dx * dx + dy * dy + dz * dz);
    const double ux = dx * in, uy = dy * in, uz = dz * in;
    const double p = v[0] * ux + v[1] * uy + v[2] * uz;
    v[0] -= p * ux;
    v[1] -= p * uy;
    v[2] -= p * uz;
}

// A magnetic first point (timedomainkernal, empropagation.py:1395-1419):
// v = Re(w) x d / eta, d the float64 unit direction a -> b
LEM_DEV void magnetic_launch(const float *__restrict__ pos, int64_t a, int64_t b, double eta,
                             double v[3])
{
    const double dx = (double)(pos[3 * b] - pos[3 * a]);
    const double dy = (double)(pos[3 * b + 1] - pos[3 * a + 1]);
    const double dz = (double)(pos[3 * b + 2] - pos[3 * a + 2]);
    const double n = sqrt(dx * dx + dy * dy + dz * dz);
    const double ux = dx / n, uy = dy / n, uz = dz / n;
    const double mx = (v[1] * uz - v[2] * uy) / eta;
    const double my = (v[2] * ux - v[0] * uz) / eta;
    const double mz = (v[0] * uy - v[1] * ux) / eta;
    v[0] = mx;
    v[1] = my;
    v[2] = mz;
}

// (I - n n^T) v with n the normalised point normal (the u/v basis of
// sourcelaunchtransformGPU is built from normalised cross products)
LEM_DEV void project_normal64(const float *__restrict__ nrm, int64_t a, double v[3])
{
    const double mx = nrm[3 * a], my = nrm[3 * a + 1], mz = nrm[3 * a + 2];
    const double im = 1.0 / sqrt(mx * mx + my * my + mz * mz);
    const double nx = mx * im, ny = my * im, nz = mz * im;
    const double p = v[0] * nx + v[1] * ny + v[2] * nz;
    v[0] -= p * nx;
    v[1] -= p * ny;
    v[2] -= p * nz;
}

__global__ __launch_bounds__(TB) void k_time_paths(
    const float *__restrict__ pos, const float *__restrict__ nrm, const float2 *__restrict__ w,
    const float *__restrict__ eta, int64_t N, const int32_t *__restrict__ index, int64_t V,
    int ncol, double alpha, double beta,
    double *__restrict__ amp, double *__restrict__ arrival, int32_t *__restrict__ err)
{
    const int64_t v = (int64_t)blockIdx.x * TB + threadIdx.x;
    if (v >= V)
        return;
    const int32_t *row = index + v * ncol;
    bool ok = row[0] != 0;
    for (int i = 0; i < ncol; ++i)
        ok = ok && row[i] >= 0 && (int64_t)row[i] <= N;
    if (!ok) {
        err[0] = 1;
        const double nan = __longlong_as_double(0x7ff8000000000000ll);
        amp[3 * v] = amp[3 * v + 1] = amp[3 * v + 2] = arrival[v] = nan;
        return;
    }
    const int64_t p0 = wrap_point(row[0], N), p1 = wrap_point(row[1], N);
    double len = sep64(pos, p0, p1);
    double delay = (double)w[3 * p0].y;
    double rc[3] = {(double)w[3 * p0].x, (double)w[3 * p0 + 1].x, (double)w[3 * p0 + 2].x};
    if (eta && eta[p0] > 0.0f)
        magnetic_launch(pos, p0, p1, (double)eta[p0], rc);
    if (row[1] != 0) {
        project_dir(pos, p0, p1, rc);
        rc[0] *= (double)w[3 * p1].x;
        rc[1] *= (double)w[3 * p1 + 1].x;
        rc[2] *= (double)w[3 * p1 + 2].x;
        delay += (double)w[3 * p1].y;
    }
    double mag = loss_mag(pos, nrm, p0, p1, alpha, beta);
    for (int i = 1; i < ncol - 1; ++i) {
        const int64_t a = wrap_point(row[i], N), b = wrap_point(row[i + 1], N);
        project_normal64(nrm, a, rc);
        len += sep64(pos, a, b);
        if (row[i + 1] != 0) {
            project_dir(pos, a, b, rc);
            rc[0] *= (double)w[3 * b].x;
            rc[1] *= (double)w[3 * b + 1].x;
            rc[2] *= (double)w[3 * b + 2].x;
            delay += (double)w[3 * b].y;
            mag *= loss_mag(pos, nrm, a, b, alpha, beta);
        }
    }
    amp[3 * v] = rc[0] * mag;
    amp[3 * v + 1] = rc[1] * mag;
    amp[3 * v + 2] = rc[2] * mag;
    arrival[v] = len / LIGHT_SPEED + delay;
}

// Order-preserving map of float64 to uint64 (for an atomic minimum).
LEM_DEV unsigned long long dkey(double d)
{
    const unsigned long long u = (unsigned long long)__double_as_longlong(d);
    return (u >> 63) ? ~u : (u | 0x8000000000000000ull);
}
LEM_DEV double dkey_inv(unsigned long long k)
{
    const unsigned long long u = (k >> 63) ? (k & 0x7fffffffffffffffull) : ~k;
    return __longlong_as_double((long long)u);
}

// Bound by the read: four loads in flight a thread, and one atomic minimum per 16
// wavefronts (16.8 M arrivals: 51 us with one load and one per 4 -> 30).
constexpr int WAKE_TB = 1024, WAKE_BLOCKS = 1024;
__global__ __launch_bounds__(WAKE_TB) void k_time_wake(const double *__restrict__ arrival,
                                                       int64_t V,
                                                       unsigned long long *__restrict__ key)
{
    __shared__ unsigned long long s[WAKE_TB / 64];
    unsigned long long m = dkey(1.0);
    const int64_t stride = (int64_t)gridDim.x * WAKE_TB;
    for (int64_t i = (int64_t)blockIdx.x * WAKE_TB + threadIdx.x; i < V; i += 4 * stride) {
        double a[4];
#pragma unroll
        for (int q = 0; q < 4; ++q)
            a[q] = i + q * stride < V ? arrival[i + q * stride] : 1.0;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (a[q] == a[q]) {  // NaN arrivals take no part
                const unsigned long long k = dkey(a[q]);
                m = k < m ? k : m;
            }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const unsigned long long k = __shfl_xor(m, off);
        m = k < m ? k : m;
    }
    if ((threadIdx.x & 63) == 0)
        s[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < WAKE_TB / 64; ++w)
            m = s[w] < m ? s[w] : m;
        atomicMin(key, m);
    }
}

__global__ void k_time_wake_init(unsigned long long *__restrict__ key)
{
    if (threadIdx.x == 0)
        *key = dkey(1.0);
}

__global__ void k_time_wake_finish(unsigned long long *__restrict__ key)
{
    if (threadIdx.x == 0)
        *reinterpret_cast<double *>(key) = dkey_inv(*key);
}

// Python's float floor division a // b (CPython float_floor_div, which numba
// follows): fmod-based, exact for the integer-valued results used as indices.
LEM_DEV double py_floordiv(double a, double b)
{
    double mod = fmod(a, b);
    double div = (a - mod) / b;
    if (mod != 0.0) {
        if ((b < 0.0) != (mod < 0.0))
            div -= 1.0;
    }
    if (div != 0.0) {
        double fl = floor(div);
        if (div - fl > 0.5)
            fl += 1.0;
        return fl;
    }
    return copysign(0.0, a / b);
}

// start sample of each path
__global__ __launch_bounds__(TB) void k_time_bins(const double *__restrict__ arrival, int64_t V,
                                                  const double *__restrict__ wake, double sep,
                                                  int64_t *__restrict__ bin)
{
    const int64_t v = (int64_t)blockIdx.x * TB + threadIdx.x;
    if (v >= V)
        return;
    const double b = py_floordiv(arrival[v] - *wake, sep);
    bin[v] = b < 9.0e18 ? (int64_t)b : (int64_t)9e18;
}

// One thread per (segment, sample n): sum over the segment's paths, in path
// order, of excitation[n - bin] * amp.  Segments are the (source, sink) slots
// (paths sorted stably by slot).  Grid: (ceil(N / TB), nseg).
__global__ __launch_bounds__(TB) void k_time_map(
    const double *__restrict__ amp, const int64_t *__restrict__ bin,
    const int64_t *__restrict__ order, const int64_t *__restrict__ seg_start,
    const int64_t *__restrict__ seg_slot, const double *__restrict__ exc, int64_t E, int64_t N,
    double *__restrict__ out)
{
    const int64_t n = (int64_t)blockIdx.x * TB + threadIdx.x;
    const int64_t g = blockIdx.y;
    if (n >= N)
        return;
    double a0 = 0.0, a1 = 0.0, a2 = 0.0;
    for (int64_t q = seg_start[g]; q < seg_start[g + 1]; ++q) {
        const int64_t p = order[q];
        const int64_t j = n - bin[p];
        if (j >= 0 && j < E) {
            const double e = exc[j];
            a0 += e * amp[3 * p];
            a1 += e * amp[3 * p + 1];
            a2 += e * amp[3 * p + 2];
        }
    }
    double *o = out + (seg_slot[g] * N + n) * 3;
    o[0] = a0;
    o[1] = a1;
    o[2] = a2;
}

// Trace, up to TRACE_PART_SAMPLES samples: the paths move once, in path order, to
// the bucket of 2^sh samples they start in (k_place_count, _groups, _buckets,
// _move), with their amplitudes, so that what follows reads memory in order;
// each workgroup of k_place_sums then orders SUMS_CH paths of a bucket by sample
// in LDS and sums them, and k_place_merge adds a bucket's chunks.  Chunks are cut
// by position, orders are stable, sums have a fixed shape: deterministic.  Paths
// that start past the trace's end are in no bucket.
//
// Bound by memory: 8 + 32 bytes of a path read and 26 written by the count and the
// move, 26 read by the sums.  The radix sort of (sample, path) that longer traces
// use reads 24-byte amplitudes one by one, a line each.  16.8 M paths, 65,536
// samples: 794 -> 435 us (count 30, move 206 = 4.7 TB/s, sums 147, merge 15,
// scans 13); 16 M paths of which 1 % start within 1,000 samples, one bucket:
// 69 ms (one wavefront added the rest) -> 215 us.  Past TRACE_PART_SAMPLES a bucket's sums no longer fit beside its
// paths in LDS.  Measured and left: chunks of 4,096 in the move (one workgroup a
// CU, 242 us) and in the sums (205), buckets of 512 samples (move 190, sums 160,
// merge 20).
constexpr int PT = 1024;         // threads
constexpr int PW = PT / 64;
constexpr int MOVE_R = 2, SUMS_R = 2;  // paths of one thread
constexpr int MOVE_CH = PT * MOVE_R, SUMS_CH = PT * SUMS_R;
constexpr int PLACE_NB = 256;    // most buckets
constexpr int PLACE_GROUP = 64;  // chunks whose counts one workgroup adds up
constexpr int PLACE_SH_MIN = 8, PLACE_SH_MAX = 10;
constexpr int PLACE_COLS = 3 << PLACE_SH_MAX >> 10;  // sums of one thread, at most
static_assert(PT == 1024, "PLACE_COLS");
constexpr int64_t TRACE_PART_SAMPLES = (int64_t)PLACE_NB << PLACE_SH_MAX;

// bucket and sample in the bucket of a start sample; -1 past the end.  Samples
// before the trace's start count as its first, as in the sort.
LEM_DEV int place_sample(int64_t b, int64_t N) { return b >= N ? -1 : (b < 0 ? 0 : (int)b); }

// rank[r]: how many earlier entries of this wavefront (rounds of 64 lanes) have the
// same digit; cnt (the wavefront's own, zero before) ends up with the digit counts.
template <int R>
LEM_DEV void wave_ranks(const int (&digit)[R], int bits, volatile uint16_t *cnt, int (&rank)[R])
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int d = digit[r];
        unsigned long long m = __ballot(d >= 0);
        for (int b = 0; b < bits; ++b) {
            const bool on = (d >> b) & 1;
            const unsigned long long v = __ballot(on);
            m &= on ? v : ~v;
        }
        if (d >= 0) {
            const int base = cnt[d];
            rank[r] = base + __popcll(m & ((1ull << lane) - 1));
            __builtin_amdgcn_wave_barrier();
            if (m >> lane == 1)
                cnt[d] = (uint16_t)(base + __popcll(m));
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// Exclusive sum over the workgroup; total: the sum of all.
LEM_DEV int block_exclusive(int x, int *s_wave, int *total)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int y = x;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int z = __shfl_up(y, off);
        y += lane >= off ? z : 0;
    }
    if (lane == 63)
        s_wave[wave] = y;
    __syncthreads();
    int before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < PW; ++w) {
        before += w < wave ? s_wave[w] : 0;
        all += s_wave[w];
    }
    *total = all;
    return before + y - x;
}

// Ranks of the workgroup's entries by digit (nd digits): place[r] = position in the
// stable order; first (of digit threadIdx.x) and *total as counted.  cnt: PW x nd.
template <int R>
LEM_DEV int block_places(const int (&digit)[R], int nd, int bits, uint16_t *cnt, int *s_wave,
                         int (&place)[R], int *total)
{
    const int wave = threadIdx.x >> 6;
    for (int i = threadIdx.x; i < PW * nd; i += PT)
        cnt[i] = 0;
    __syncthreads();
    wave_ranks(digit, bits, cnt + wave * nd, place);
    __syncthreads();
    int n = 0;
    if ((int)threadIdx.x < nd)
        for (int w = 0; w < PW; ++w)
            n += cnt[w * nd + threadIdx.x];
    const int first = block_exclusive(n, s_wave, total);
    if ((int)threadIdx.x < nd) {
        int at = first;
        for (int w = 0; w < PW; ++w) {
            const int c = cnt[w * nd + threadIdx.x];
            cnt[w * nd + threadIdx.x] = (uint16_t)at;  // at < 64 R PW where c > 0
            at += c;
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r)
        if (digit[r] >= 0)
            place[r] += cnt[wave * nd + digit[r]];
    return first;
}

// entry r of this thread: the chunk in rounds of 64 lanes, wavefront by wavefront
template <int R>
LEM_DEV int place_entry(int r)
{
    return (threadIdx.x >> 6) * (64 * R) + r * 64 + (threadIdx.x & 63);
}

// counts[chunk][bucket]
__global__ __launch_bounds__(PT) void k_place_count(const int64_t *__restrict__ bin, int64_t V,
                                                    int64_t N, int sh, int *__restrict__ counts)
{
    __shared__ int s_n[PLACE_NB];
    if (threadIdx.x < PLACE_NB)
        s_n[threadIdx.x] = 0;
    __syncthreads();
    const int64_t c0 = (int64_t)blockIdx.x * MOVE_CH;
#pragma unroll
    for (int r = 0; r < MOVE_R; ++r) {
        const int64_t v = c0 + r * PT + threadIdx.x;
        const int k = v < V ? place_sample(bin[v], N) : -1;
        if (k >= 0)
            atomicAdd(&s_n[k >> sh], 1);
    }
    __syncthreads();
    if (threadIdx.x < PLACE_NB)
        counts[(int64_t)blockIdx.x * PLACE_NB + threadIdx.x] = s_n[threadIdx.x];
}

// counts -> the paths of the bucket in earlier chunks of the group; sums[group][bucket]
__global__ __launch_bounds__(PLACE_NB) void k_place_groups(int *__restrict__ counts,
                                                           int64_t nchunk, int *__restrict__ sums)
{
    const int64_t c0 = (int64_t)blockIdx.x * PLACE_GROUP;
    const int64_t c1 = c0 + PLACE_GROUP < nchunk ? c0 + PLACE_GROUP : nchunk;
    int at = 0;
#pragma unroll 8
    for (int64_t c = c0; c < c1; ++c) {
        const int n = counts[c * PLACE_NB + threadIdx.x];
        counts[c * PLACE_NB + threadIdx.x] = at;
        at += n;
    }
    sums[(int64_t)blockIdx.x * PLACE_NB + threadIdx.x] = at;
}

// sums -> the bucket's first position plus its paths in earlier groups.
// first[b]: bucket b's first position, chunk[b]: chunks of buckets before b.
__global__ __launch_bounds__(PT) void k_place_buckets(int *__restrict__ sums, int64_t ngroup,
                                                      int *__restrict__ first,
                                                      int *__restrict__ chunk)
{
    __shared__ int s_part[PW * 64], s_wave[PW];
    // PLACE_Q threads a bucket, each a share of the groups
    const int b = threadIdx.x & (PLACE_NB - 1), q = threadIdx.x / PLACE_NB;
    constexpr int PLACE_Q = PT / PLACE_NB;
    const int64_t g0 = ngroup * q / PLACE_Q, g1 = ngroup * (q + 1) / PLACE_Q;
    int n = 0;
#pragma unroll 4
    for (int64_t g = g0; g < g1; ++g)
        n += sums[g * PLACE_NB + b];
    s_part[q * PLACE_NB + b] = n;
    __syncthreads();
    int all = 0, before = 0;
    for (int i = 0; i < PLACE_Q; ++i) {
        all += s_part[i * PLACE_NB + b];
        before += i < q ? s_part[i * PLACE_NB + b] : 0;
    }
    int total, chunks;
    const int f = block_exclusive(q == 0 ? all : 0, s_wave, &total);
    __syncthreads();
    const int c = block_exclusive(q == 0 ? (int)(((int64_t)all + SUMS_CH - 1) / SUMS_CH) : 0,
                                  s_wave, &chunks);
    __syncthreads();
    if (q == 0) {
        s_part[b] = f;
        first[b] = f;
        chunk[b] = c;
        if (b == 0) {
            first[PLACE_NB] = total;
            chunk[PLACE_NB] = chunks;
        }
    }
    __syncthreads();
    int at = s_part[b] + before;
#pragma unroll 4
    for (int64_t g = g0; g < g1; ++g) {
        const int k = sums[g * PLACE_NB + b];
        sums[g * PLACE_NB + b] = at;
        at += k;
    }
}

constexpr int PLACE_MOVE_LDS = MOVE_CH * (24 + 2 + 2) + PW * PLACE_NB * 2 + PLACE_NB * 4 + PW * 4;

__global__ __launch_bounds__(PT) void k_place_move(
    const int64_t *__restrict__ bin, const double *__restrict__ amp, int64_t V, int64_t N, int sh,
    const int *__restrict__ counts, const int *__restrict__ sums, uint16_t *__restrict__ key,
    double *__restrict__ moved)
{
    extern __shared__ __align__(16) char s_mem[];
    double *s_amp = reinterpret_cast<double *>(s_mem);
    uint16_t *s_key = reinterpret_cast<uint16_t *>(s_mem + MOVE_CH * 24);
    uint16_t *s_bucket = s_key + MOVE_CH;
    uint16_t *s_cnt = s_bucket + MOVE_CH;
    int *s_to = reinterpret_cast<int *>(s_cnt + PW * PLACE_NB);
    int *s_wave = s_to + PLACE_NB;
    // an XCD takes consecutive chunks: the runs that share a line share its L2
    const int64_t nchunk = (V + MOVE_CH - 1) / MOVE_CH;
    const int64_t chunk = (blockIdx.x & 7) * ((nchunk + 7) / 8) + (blockIdx.x >> 3);
    if (chunk >= nchunk)
        return;
    const int64_t c0 = chunk * MOVE_CH;
    int digit[MOVE_R], local[MOVE_R], place[MOVE_R];
    double a[MOVE_R][3];
#pragma unroll
    for (int r = 0; r < MOVE_R; ++r) {
        const int64_t v = c0 + place_entry<MOVE_R>(r);
        const int k = v < V ? place_sample(bin[v], N) : -1;
        digit[r] = k >> sh;  // -1 stays -1
        local[r] = k & ((1 << sh) - 1);
    }
#pragma unroll
    for (int r = 0; r < MOVE_R; ++r)
        if (digit[r] >= 0) {
            const int64_t v = c0 + place_entry<MOVE_R>(r);
#pragma unroll
            for (int c = 0; c < 3; ++c)
                a[r][c] = amp[3 * v + c];
        }
    int n;
    const int f = block_places(digit, PLACE_NB, 8, s_cnt, s_wave, place, &n);
    if (threadIdx.x < PLACE_NB)
        s_to[threadIdx.x] = counts[chunk * PLACE_NB + threadIdx.x] +
                            sums[(chunk / PLACE_GROUP) * PLACE_NB + threadIdx.x] - f;
#pragma unroll
    for (int r = 0; r < MOVE_R; ++r)
        if (digit[r] >= 0) {
            s_key[place[r]] = (uint16_t)local[r];
            s_bucket[place[r]] = (uint16_t)digit[r];
#pragma unroll
            for (int c = 0; c < 3; ++c)
                s_amp[3 * place[r] + c] = a[r][c];
        }
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += PT)
        key[(int64_t)s_to[s_bucket[i]] + i] = s_key[i];
    for (int i = threadIdx.x; i < 3 * n; i += PT) {
        const int p = i / 3;
        moved[((int64_t)s_to[s_bucket[p]] + p) * 3 + (i - 3 * p)] = s_amp[i];
    }
}

inline int place_sums_lds(int sh) { return SUMS_CH * 24 + ((PW * 2) << sh) + (1 << sh) * 2 + 8 + PW * 4; }

// Sums of one chunk: part[chunk][sample of the bucket][3].  DIRECT: the trace is one
// bucket, nothing was moved (key: none), and a workgroup adds up `per` chunks in
// path order.
template <bool DIRECT>
__global__ __launch_bounds__(PT) void k_place_sums(
    const int64_t *__restrict__ bin, const uint16_t *__restrict__ key,
    const double *__restrict__ amp, int64_t V, int64_t N, int sh, const int *__restrict__ first,
    const int *__restrict__ chunk, int64_t per, double *__restrict__ part)
{
    extern __shared__ __align__(16) char s_mem[];
    double *s_amp = reinterpret_cast<double *>(s_mem);
    const int nd = 1 << sh, cols = 3 * nd;
    uint16_t *s_cnt = reinterpret_cast<uint16_t *>(s_mem + SUMS_CH * 24);
    uint16_t *s_first = s_cnt + PW * nd;  // nd + 1 of them
    int *s_wave = reinterpret_cast<int *>(s_first + nd + 2);
    int64_t v0, v1;
    if (DIRECT) {
        v0 = (int64_t)blockIdx.x * per * SUMS_CH;
        v1 = v0 + per * SUMS_CH < V ? v0 + per * SUMS_CH : V;
    } else {
        if ((int)blockIdx.x >= chunk[PLACE_NB])
            return;
        int lo = 0, hi = PLACE_NB;  // last bucket with chunk[b] <= id (buckets may be empty)
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (chunk[mid] <= (int)blockIdx.x)
                lo = mid;
            else
                hi = mid;
        }
        v0 = (int64_t)first[lo] + (int64_t)((int)blockIdx.x - chunk[lo]) * SUMS_CH;
        v1 = first[lo + 1];
    }
    double sum[PLACE_COLS] = {};
    do {
        int digit[SUMS_R], place[SUMS_R];
        double a[SUMS_R][3];
#pragma unroll
        for (int r = 0; r < SUMS_R; ++r) {
            const int64_t v = v0 + place_entry<SUMS_R>(r);
            digit[r] = -1;
            if (v < v1)
                digit[r] = DIRECT ? place_sample(bin[v], N) : (int)key[v];
            if (digit[r] >= 0) {
#pragma unroll
                for (int c = 0; c < 3; ++c)
                    a[r][c] = amp[3 * v + c];
            }
        }
        int n;
        const int f = block_places(digit, nd, sh, s_cnt, s_wave, place, &n);
        if ((int)threadIdx.x < nd)
            s_first[threadIdx.x] = (uint16_t)f;
        if (threadIdx.x == 0)
            s_first[nd] = (uint16_t)n;
#pragma unroll
        for (int r = 0; r < SUMS_R; ++r)
            if (digit[r] >= 0)
#pragma unroll
                for (int c = 0; c < 3; ++c)
                    s_amp[3 * place[r] + c] = a[r][c];
        __syncthreads();
#pragma unroll
        for (int q = 0; q < PLACE_COLS; ++q) {
            const int i = q * PT + threadIdx.x;
            if (i >= cols)
                break;
            const int d = i / 3, c = i - 3 * d;
            const int e = s_first[d + 1];
            for (int p = s_first[d]; p < e; ++p)
                sum[q] += s_amp[3 * p + c];
        }
        if (!DIRECT)
            break;
        v0 += SUMS_CH;
        __syncthreads();
    } while (v0 < v1);
    double *out = part + (int64_t)blockIdx.x * cols;
#pragma unroll
    for (int q = 0; q < PLACE_COLS; ++q)
        if (q * PT + (int)threadIdx.x < cols)
            out[q * PT + threadIdx.x] = sum[q];
}

// H of a bucket: its chunks' sums, 16 strided shares and then those in order.
// Grid: (ceil(3 * 2^sh / 64), buckets).
__global__ __launch_bounds__(PT) void k_place_merge(const double *__restrict__ part,
                                                    const int *__restrict__ chunk, int64_t direct,
                                                    int64_t N, int sh, double *__restrict__ H)
{
    __shared__ double s[PW][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int cols = 3 << sh, col = blockIdx.x * 64 + lane, b = blockIdx.y;
    const int64_t c0 = chunk ? chunk[b] : 0, c1 = chunk ? chunk[b + 1] : direct;
    double h = 0.0;
    if (col < cols) {
#pragma unroll 4
        for (int64_t c = c0 + wave; c < c1; c += PW)
            h += part[c * cols + col];
    }
    s[wave][lane] = h;
    __syncthreads();
    const int64_t at = (int64_t)b * cols + col;
    if (wave == 0 && col < cols && at < 3 * N) {
#pragma unroll
        for (int w = 1; w < PW; ++w)
            h += s[w][lane];
        H[at] = h;
    }
}

// Longer traces: sort keys (start sample clamped to [0, N]; N = never placed).
__global__ __launch_bounds__(TB) void k_trace_keys(const int64_t *__restrict__ bin, int64_t V,
                                                   int64_t N, int32_t *__restrict__ key,
                                                   int32_t *__restrict__ val)
{
    const int64_t p = (int64_t)blockIdx.x * TB + threadIdx.x;
    if (p >= V)
        return;
    const int64_t b = bin[p];
    key[p] = (int32_t)(b < 0 ? 0 : (b >= N ? N : b));
    val[p] = (int32_t)p;
}

// start[b] = first sorted position with key >= b, for b in [0, N]
__global__ __launch_bounds__(TB) void k_trace_starts(const int32_t *__restrict__ key, int64_t V,
                                                     int64_t N, int32_t *__restrict__ start)
{
    const int64_t b = (int64_t)blockIdx.x * TB + threadIdx.x;
    if (b > N)
        return;
    int64_t lo = 0, hi = V;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (key[mid] < b)
            lo = mid + 1;
        else
            hi = mid;
    }
    start[b] = (int32_t)lo;
}

// H[b] = sum of the amplitudes of the paths starting at sample b.  One
// wavefront per sample: lane l sums the sample's paths l, l + 64, ... in path
// order, then the 64 partial sums meet in a fixed butterfly -- the order is
// fixed, so the result is deterministic.
__global__ __launch_bounds__(TB) void k_trace_hist(const double *__restrict__ amp,
                                                   const int32_t *__restrict__ val,
                                                   const int32_t *__restrict__ start, int64_t N,
                                                   double *__restrict__ H)
{
    const int64_t b = (int64_t)blockIdx.x * (TB / 64) + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (b >= N)
        return;  // wave-uniform
    double h0 = 0.0, h1 = 0.0, h2 = 0.0;
    const int32_t e = start[b + 1];
    for (int32_t i = start[b] + lane; i < e; i += 64) {
        const int64_t p = val[i];
        h0 += amp[3 * p];
        h1 += amp[3 * p + 1];
        h2 += amp[3 * p + 2];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        h0 += __shfl_xor(h0, off);
        h1 += __shfl_xor(h1, off);
        h2 += __shfl_xor(h2, off);
    }
    if (lane == 0) {
        H[3 * b] = h0;
        H[3 * b + 1] = h1;
        H[3 * b + 2] = h2;
    }
}

// out[n] = sum_{j <= min(E - 1, n)} exc[j] H[n - j]: 64 samples a workgroup, its 16
// wavefronts take a share of the excitation each and the shares are added in order
// (one wavefront a SIMD with all of it, 65,536 samples and 256 of excitation: 36 us;
// this: 18).
__global__ __launch_bounds__(PT) void k_trace_conv(const double *__restrict__ H,
                                                   const double *__restrict__ exc, int64_t E,
                                                   int64_t N, double *__restrict__ out)
{
    __shared__ double s[PW][3][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t n = (int64_t)blockIdx.x * 64 + lane;
    const int64_t share = (E + PW - 1) / PW;
    const int64_t j0 = wave * share;
    int64_t j1 = j0 + share < E ? j0 + share : E;
    j1 = n < N ? (j1 < n + 1 ? j1 : n + 1) : 0;
    double a0 = 0.0, a1 = 0.0, a2 = 0.0;
#pragma unroll 4
    for (int64_t j = j0; j < j1; ++j) {
        const double e = exc[j];
        const double *h = H + 3 * (n - j);
        a0 += e * h[0];
        a1 += e * h[1];
        a2 += e * h[2];
    }
    s[wave][0][lane] = a0;
    s[wave][1][lane] = a1;
    s[wave][2][lane] = a2;
    __syncthreads();
    if (threadIdx.x < 192) {
        const int64_t at = (int64_t)blockIdx.x * 192 + threadIdx.x;
        const int i = threadIdx.x / 3, c = threadIdx.x - 3 * i;
        double a = 0.0;
#pragma unroll
        for (int w = 0; w < PW; ++w)
            a += s[w][c][i];
        if (at < 3 * N)
            out[at] = a;
    }
}

struct TraceWs {
    int32_t *k0, *k1, *v0, *v1, *start;
    int *counts, *sums, *first, *chunk;
    uint16_t *key;
    double *moved, *part, *H;
    void *cub;
    size_t cub_bytes;
};

inline int key_bits(int64_t N)
{
    int b = 1;
    while (b < 31 && ((int64_t)1 << b) <= N)
        ++b;
    return b;
}

inline int64_t align256(int64_t x) { return (x + 255) / 256 * 256; }

// log2 of a bucket's samples: as few as cover the trace, which keeps the chunks' sums
// short; a trace of at most 2^PLACE_SH_MAX samples is one bucket and nothing moves.
inline int place_shift(int64_t N)
{
    int sh = PLACE_SH_MIN;
    while (sh < PLACE_SH_MAX && ((int64_t)PLACE_NB << sh) < N)
        ++sh;
    while (N <= ((int64_t)1 << PLACE_SH_MAX) && ((int64_t)1 << sh) < N)
        ++sh;
    return sh;
}

// Workgroups of k_place_sums<true>: four a CU or as many as there are chunks.
inline int64_t place_direct(int64_t V) { return std::min<int64_t>(ceil_div(V, SUMS_CH), 1024); }

// Lays the trace workspace out from base (or only sizes it when base is null).
inline int64_t trace_layout(int64_t V, int64_t N, size_t cub_bytes, char *base, TraceWs *L)
{
    int64_t off = 0;
    auto take = [&](int64_t bytes) {
        char *p = base ? base + off : nullptr;
        off += align256(bytes);
        return p;
    };
    TraceWs l = {};
    l.H = reinterpret_cast<double *>(take(8 * 3 * N));
    if (N <= TRACE_PART_SAMPLES) {
        const int sh = place_shift(N);
        const int64_t nchunk = ceil_div(V, MOVE_CH);
        const bool direct = N <= ((int64_t)1 << sh);
        l.part = reinterpret_cast<double *>(
            take((direct ? place_direct(V) : ceil_div(V, SUMS_CH) + PLACE_NB) * (24LL << sh)));
        if (!direct) {
            l.counts = reinterpret_cast<int *>(take(4 * PLACE_NB * nchunk));
            l.sums = reinterpret_cast<int *>(take(4 * PLACE_NB * ceil_div(nchunk, PLACE_GROUP)));
            l.first = reinterpret_cast<int *>(take(4 * (PLACE_NB + 1)));
            l.chunk = reinterpret_cast<int *>(take(4 * (PLACE_NB + 1)));
            l.key = reinterpret_cast<uint16_t *>(take(2 * V));
            l.moved = reinterpret_cast<double *>(take(24 * V));
        }
    } else {
        l.k0 = reinterpret_cast<int32_t *>(take(4 * V));
        l.k1 = reinterpret_cast<int32_t *>(take(4 * V));
        l.v0 = reinterpret_cast<int32_t *>(take(4 * V));
        l.v1 = reinterpret_cast<int32_t *>(take(4 * V));
        l.start = reinterpret_cast<int32_t *>(take(4 * (N + 2)));
        l.cub = take((int64_t)cub_bytes);
        l.cub_bytes = cub_bytes;
    }
    if (L)
        *L = l;
    return off;
}

// Scratch bytes of the radix sort, or -1 when the size query fails.
inline int64_t cub_sort_bytes(int64_t V, int64_t N)
{
    size_t bytes = 0;
    if (hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, (const int32_t *)nullptr,
                                           (int32_t *)nullptr, (const int32_t *)nullptr,
                                           (int32_t *)nullptr, (int)V, 0,
                                           key_bits(N)) != hipSuccess)
        return -1;
    return (int64_t)bytes;
}

}  // namespace lem

using namespace lem;

extern "C" int lem_time_paths(const float *pos, const float *nrm, const float *w,
                              const float *eta, int64_t N,
                              const int32_t *index, int64_t V, int ncol, double alpha, double beta,
                              double *amp, double *arrival, int32_t *err, void *stream)
{
    clear_error();
    LEM_REQUIRE(ncol >= 2 && ncol <= 8, "lem_time_paths: index needs 2 to 8 columns");
    LEM_REQUIRE(V >= 0 && N >= 0, "lem_time_paths: negative size");
    if (V == 0)
        return 0;
    LEM_REQUIRE(N > 0 && pos && nrm && w && index && amp && arrival && err,
                "lem_time_paths: null pointer");
    hipLaunchKernelGGL(k_time_paths, dim3((unsigned)ceil_div(V, TB)), dim3(TB), 0,
                       as_stream(stream), pos, nrm, reinterpret_cast<const float2 *>(w), eta, N,
                       index, V, ncol, alpha, beta, amp, arrival, err);
    return check_launch("k_time_paths");
}

extern "C" int lem_time_wake(const double *arrival, int64_t V, double *wake, void *stream)
{
    clear_error();
    LEM_REQUIRE(V >= 0 && wake && (V == 0 || arrival), "lem_time_wake: bad arguments");
    hipStream_t st = as_stream(stream);
    unsigned long long *key = reinterpret_cast<unsigned long long *>(wake);
    hipLaunchKernelGGL(k_time_wake_init, dim3(1), dim3(64), 0, st, key);
    if (V > 0) {
        const int64_t nb = std::min<int64_t>(ceil_div(V, WAKE_TB), WAKE_BLOCKS);
        hipLaunchKernelGGL(k_time_wake, dim3((unsigned)nb), dim3(WAKE_TB), 0, st, arrival, V, key);
    }
    hipLaunchKernelGGL(k_time_wake_finish, dim3(1), dim3(64), 0, st, key);
    return check_launch("k_time_wake");
}

extern "C" int lem_time_bins(const double *arrival, int64_t V, const double *wake,
                             double sampling_freq, int64_t *bin, void *stream)
{
    clear_error();
    LEM_REQUIRE(V >= 0 && sampling_freq > 0.0, "lem_time_bins: bad arguments");
    if (V == 0)
        return 0;
    LEM_REQUIRE(arrival && wake && bin, "lem_time_bins: null pointer");
    hipLaunchKernelGGL(k_time_bins, dim3((unsigned)ceil_div(V, TB)), dim3(TB), 0,
                       as_stream(stream), arrival, V, wake, 1.0 / sampling_freq, bin);
    return check_launch("k_time_bins");
}

extern "C" int lem_time_map(const double *amp, const int64_t *bin, const int64_t *order,
                            const int64_t *seg_start, const int64_t *seg_slot, int64_t nseg,
                            const double *excitation, int64_t E, int64_t N, double *out,
                            void *stream)
{
    clear_error();
    LEM_REQUIRE(nseg >= 0 && E >= 0 && N >= 0, "lem_time_map: negative size");
    if (nseg == 0 || N == 0)
        return 0;
    LEM_REQUIRE(amp && bin && order && seg_start && seg_slot && out && (E == 0 || excitation),
                "lem_time_map: null pointer");
    // at most 65535 segments per launch (grid y)
    for (int64_t g0 = 0; g0 < nseg; g0 += 65535) {
        const int64_t ng = std::min<int64_t>(nseg - g0, 65535);
        dim3 grid((unsigned)ceil_div(N, TB), (unsigned)ng);
        hipLaunchKernelGGL(k_time_map, grid, dim3(TB), 0, as_stream(stream), amp, bin, order,
                           seg_start + g0, seg_slot + g0, excitation, E, N, out);
        const int rc = check_launch("k_time_map");
        if (rc)
            return rc;
    }
    return 0;
}

extern "C" int64_t lem_time_trace_workspace(int64_t V, int64_t N)
{
    if (V < 0 || N < 0 || V > 2000000000LL || N > 2000000000LL)
        return -1;
    const int64_t cub = N > TRACE_PART_SAMPLES ? cub_sort_bytes(V > 0 ? V : 1, N) : 0;
    if (cub < 0)
        return -1;
    return trace_layout(V > 0 ? V : 1, N, (size_t)cub, nullptr, nullptr);
}

extern "C" int lem_time_trace(const double *amp, const int64_t *bin, int64_t V,
                              const double *excitation, int64_t E, int64_t N, double *out,
                              void *workspace, int64_t workspace_bytes, void *stream)
{
    clear_error();
    LEM_REQUIRE(V >= 0 && E >= 0 && N >= 0, "lem_time_trace: negative size");
    LEM_REQUIRE(V <= 2000000000LL && N <= 2000000000LL, "lem_time_trace: too many paths or samples");
    if (N == 0)
        return 0;
    LEM_REQUIRE(out && (V == 0 || (amp && bin)) && (E == 0 || excitation),
                "lem_time_trace: null pointer");
    LEM_REQUIRE(ceil_div(N, TB / 64) <= 2147483647LL, "lem_time_trace: too many samples");
    const int64_t Vs = V > 0 ? V : 1;
    const int64_t cub = N > TRACE_PART_SAMPLES ? cub_sort_bytes(Vs, N) : 0;
    if (cub < 0) {
        set_error("lem_time_trace: radix sort size query failed");
        return E_HIP;
    }
    const size_t cub_bytes = (size_t)cub;
    const int64_t need = trace_layout(Vs, N, cub_bytes, nullptr, nullptr);
    if (!workspace || workspace_bytes < need) {
        set_error("lem_time_trace: workspace smaller than lem_time_trace_workspace()");
        return E_WORKSPACE;
    }
    TraceWs L;
    trace_layout(Vs, N, cub_bytes, reinterpret_cast<char *>(workspace), &L);
    hipStream_t st = as_stream(stream);
    int rc = 0;
    if (N <= TRACE_PART_SAMPLES) {
        const int sh = place_shift(N);
        const int64_t nchunk = ceil_div(V, MOVE_CH), ngroup = ceil_div(nchunk, PLACE_GROUP);
        const int64_t nsum = ceil_div(V, SUMS_CH);
        const bool direct = N <= ((int64_t)1 << sh);
        if (nchunk > 0 && direct) {
            hipLaunchKernelGGL(k_place_sums<true>, dim3((unsigned)place_direct(V)), dim3(PT),
                               place_sums_lds(sh), st, bin, nullptr, amp, V, N, sh, nullptr,
                               nullptr, ceil_div(nsum, place_direct(V)), L.part);
        } else if (!direct) {
            if (nchunk > 0) {
                hipLaunchKernelGGL(k_place_count, dim3((unsigned)nchunk), dim3(PT), 0, st, bin, V,
                                   N, sh, L.counts);
                hipLaunchKernelGGL(k_place_groups, dim3((unsigned)ngroup), dim3(PLACE_NB), 0, st,
                                   L.counts, nchunk, L.sums);
            }
            hipLaunchKernelGGL(k_place_buckets, dim3(1), dim3(PT), 0, st, L.sums, ngroup, L.first,
                               L.chunk);
            if (nchunk > 0) {
                hipLaunchKernelGGL(k_place_move, dim3((unsigned)(8 * ceil_div(nchunk, 8))), dim3(PT), PLACE_MOVE_LDS,
                                   st, bin, amp, V, N, sh, L.counts, L.sums, L.key, L.moved);
                hipLaunchKernelGGL(k_place_sums<false>, dim3((unsigned)(nsum + PLACE_NB)),
                                   dim3(PT), place_sums_lds(sh), st, nullptr, L.key, L.moved, V, N,
                                   sh, L.first, L.chunk, 1, L.part);
            }
        }
        const dim3 mg((unsigned)ceil_div((int64_t)3 << sh, 64), (unsigned)ceil_div(N, (int64_t)1 << sh));
        hipLaunchKernelGGL(k_place_merge, mg, dim3(PT), 0, st, L.part, direct ? nullptr : L.chunk,
                           place_direct(V), N, sh, L.H);
        rc = check_launch("k_place_merge");
    } else {
        if (V > 0) {
            hipLaunchKernelGGL(k_trace_keys, dim3((unsigned)ceil_div(V, TB)), dim3(TB), 0, st, bin,
                               V, N, L.k0, L.v0);
            rc = check_launch("k_trace_keys");
            if (rc)
                return rc;
            size_t tb = L.cub_bytes;
            if (hipcub::DeviceRadixSort::SortPairs(L.cub, tb, L.k0, L.k1, L.v0, L.v1, (int)V, 0,
                                                   key_bits(N), st) != hipSuccess) {
                set_error("lem_time_trace: radix sort failed");
                return E_HIP;
            }
        }
        hipLaunchKernelGGL(k_trace_starts, dim3((unsigned)ceil_div(N + 1, TB)), dim3(TB), 0, st,
                           L.k1, V, N, L.start);
        hipLaunchKernelGGL(k_trace_hist, dim3((unsigned)ceil_div(N, TB / 64)), dim3(TB), 0, st,
                           amp, L.v1, L.start, N, L.H);
        rc = check_launch("k_trace_hist");
    }
    if (rc)
        return rc;
    hipLaunchKernelGGL(k_trace_conv, dim3((unsigned)ceil_div(N, 64)), dim3(PT), 0, st, L.H,
                       excitation, E, N, out);
    return check_launch("k_trace_conv");
}
