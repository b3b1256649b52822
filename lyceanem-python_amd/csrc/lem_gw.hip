// lem_gw.hip -- batched-excitation contraction E = G . W on MFMA (gfx950).
//
// For many excitation sets at once (the reference evaluates one excitation per
// calculate_scattering call; its multiE branch cannot run,
// frequency_domain.py:612-617), the source sum of the line-of-sight field is a
// complex matrix product per frequency f and field component c:
//
//   E[f,c,k,b] = sum_s G_c[k,s,f] W[f,s,b]
//   G_c[k,s,f] = F_f(r) (d . n_k) (e - d (d . e))_c          (all paths visible)
//
// with the lossy_propagation factor F_f (empropagation.py:768-801) at
// wavenumber k_f, d = (p_k - p_s)/r and a fixed source polarisation e.
//
// FP32 matrix instructions run at 1/16 of the bfloat16 rate, so both factors are
// split into three bfloat16 parts, x = x1 + x2 + x3 exactly (x1 and x2 rounded to
// nearest: |x2| <= 2^-8, |x3| <= 2^-17 for 1 <= |x| < 2; full float32 range, no
// scaling), and the six products x1 y1, x1 y2, x2 y1, x2 y2, x1 y3, x3 y1 accumulate in
// float32 with v_mfma_f32_32x32x16_bf16; the three left out are at most 2^-24 of x y
// together and of either sign.  The matrix instructions' own accumulation does not
// round to nearest, so the five small products have sums of their own and a step of 16
// sources is added up with ordinary float32 additions (gw_products).
// Errors, in brackets those of FP32 instructions: of one source's products against
// float64, 2.6e-8 (3.1e-8; parts cut off instead of rounded, in one chain: 7.0e-8 and
// always towards zero); of the sum of 1 / 16 / 1,024 sources, G included, 1.60e-7 /
// 1.90e-7 / 2.03e-7 (1.61e-7 / 2.08e-7 / 8.2e-7).
//
// Per step 72 matrix instructions (2,304 cycles) multiply a tile of 32 sinks x 32
// sets x 3 components, and preparing it takes about 500 vector instructions: what
// bounds both kernels below is that the two only overlap between wavefronts of a
// SIMD, of which the 96 sums and 48 partial ones leave room for two.  64 x 64
// sources, 16,384 sinks, 16 frequencies: 13.85 ms (FP32 instructions) -> 8.77 ms;
// 32 x 32 sources, 2,720 sinks, one frequency: 188 -> 73 us.  (Measured and
// left: pairs of wavefronts that share G in LDS, 9.3 ms and 98 us; matrix and vector
// instructions interleaved in one wavefront, 12 ms and more, with registers spilled;
// all six products in one chain, 8.48 ms and 74 us with an error of 3.4e-8.)
#include "lem_device.h"
#include "lem_internal.h"
#include "../../include/lem.h"

namespace lem {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int GW_M = 32;    // sinks per wavefront
constexpr int GW_B = 64;    // weight sets (columns)
constexpr int GW_N = 32;    // weight sets per wavefront
constexpr int GW_KC = 16;   // sources per step
constexpr int GW_MAX_WAVES = 8;
constexpr int GW_PLANES = 18;  // 3 components, re and im, 3 parts

// The G factor of one source -> sink path: L = F(r) (d . n) complex and the real
// projected polarisation p = e - d (d . e); G_c = L p_c.
struct GwPair {
    float Lr, Li, px, py, pz;
};

template <bool LOSSY>
LEM_DEV GwPair gw_pair(float xs, float ys, float zs, double xk, double yk, double zk, float nx,
                       float ny, float nz, float ex, float ey, float ez, double kw, double alpha)
{
#pragma clang fp contract(fast)
    const float FRONT = -0.15915494309189535f;
    const double dx = xk - (double)xs, dy = yk - (double)ys, dz = zk - (double)zs;
    const Phase p = phase_of(dx, dy, dz, kw);
    const float ir = p.inv_r;
    const float ux = (float)dx * ir, uy = (float)dy * ir, uz = (float)dz * ir;
    const float cs = ux * nx + uy * ny + uz * nz;
    float amp = ir;
    if (LOSSY)
        amp *= expf((float)(-alpha * p.r));  // rounded once: alpha r may be large
    const float Gr = amp * p.c, Gi = amp * p.s;
    const float ar = -(float)alpha - ir, ai = -(float)kw;
    const float f_ = FRONT * cs;
    const float ue = ux * ex + uy * ey + uz * ez;
    GwPair g;
    g.Lr = (ar * Gr - ai * Gi) * f_;
    g.Li = (ar * Gi + ai * Gr) * f_;
    g.px = ex - ux * ue;
    g.py = ey - uy * ue;
    g.pz = ez - uz * ue;
    return g;
}

// Three bfloat16 planes of 8 values.
struct Planes {
    bf16x8 h[3];
};

LEM_DEV uint32_t bits_of(float x) { return __builtin_bit_cast(uint32_t, x); }
// a and b rounded to bfloat16, in one word (a in the low half)
LEM_DEV uint32_t rounded_pair(float a, float b)
{
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, bf16x2));
}
LEM_DEV float low_of(uint32_t w) { return __builtin_bit_cast(float, w << 16); }
LEM_DEV float high_of(uint32_t w) { return __builtin_bit_cast(float, w & 0xffff0000u); }

// the three parts of a and b, packed; the third are what is left, 8 bits at most
LEM_DEV void split3(float a, float b, uint32_t &w0, uint32_t &w1, uint32_t &w2)
{
    w0 = rounded_pair(a, b);
    const float a2 = a - low_of(w0), b2 = b - high_of(w0);
    w1 = rounded_pair(a2, b2);
    const float a3 = a2 - low_of(w1), b3 = b2 - high_of(w1);
    w2 = __builtin_amdgcn_perm(bits_of(b3), bits_of(a3), 0x07060302u);
}

LEM_DEV f32x16 mma(const bf16x8 &a, const bf16x8 &b, const f32x16 &c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// One component's 24 products: r = gr wr - gi wi, i = gr wi + gi wr.  They start from
// zero and are added with ordinary additions: the matrix instructions' own accumulation
// does not round to nearest (chained over 4,096 sources it left an error of 1.2e-5).
// The large products x1 y1 stand apart from the small ones, the smallest of which come
// first, so that a product is cut at its own last place once; one pair of them at a
// time, for the registers (both at once, or the sums of two components pending in
// k_gw_tile, spill up to 36: 11 to 12.6 ms instead of 8.78).
LEM_DEV void gw_products(const Planes &gr, const Planes &gi, const Planes &wr, const Planes &wi,
                         const Planes &nwi, f32x16 &r, f32x16 &i)
{
    constexpr int A[5] = {0, 2, 1, 0, 1}, B[5] = {2, 0, 1, 1, 0};
    const f32x16 zero = {};
    r = zero;
    i = zero;
#pragma unroll
    for (int q = 0; q < 5; ++q) {
        r = mma(gr.h[A[q]], wr.h[B[q]], r);
        i = mma(gr.h[A[q]], wi.h[B[q]], i);
        r = mma(gi.h[A[q]], nwi.h[B[q]], r);
        i = mma(gi.h[A[q]], wr.h[B[q]], i);
    }
    __builtin_amdgcn_sched_barrier(0);
    f32x16 large = mma(gr.h[0], wr.h[0], zero);
    large = mma(gi.h[0], nwi.h[0], large);
    r += large;
    __builtin_amdgcn_sched_barrier(0);
    large = mma(gr.h[0], wi.h[0], zero);
    large = mma(gi.h[0], wr.h[0], large);
    i += large;
}

LEM_DEV bf16x8 flipped(const bf16x8 &x)
{
    return __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, x) ^ 0x80008000u);
}

// A 32 sinks x 32 sets tile.  An infinite or NaN weight, or products beyond
// float32: the parts of the split multiply infinities by zeros, so such a tile is
// done again with the FP32 instructions, which give what float32 arithmetic
// gives.  Then it is written.  k: this lane's sink (row lane % 32) for the G
// factors; k0 the tile's first.
template <bool LOSSY>
LEM_DEV void gw_finish(f32x16 (&re)[3], f32x16 (&im)[3], const float *__restrict__ src, int64_t S,
                       const float *__restrict__ snk, const float *__restrict__ snk_n, int64_t K,
                       int64_t k0, float ex, float ey, float ez, double kw, double alpha,
                       const float2 *__restrict__ Wf, float2 *__restrict__ out, int col, int64_t f)
{
    const int lane = threadIdx.x & 63, half = lane >> 5;
    float zero = 0.0f;  // stays zero if every sum is finite
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int j = 0; j < 16; ++j)
            zero = __builtin_fmaf(re[c][j], 0.0f, __builtin_fmaf(im[c][j], 0.0f, zero));
    if (__ballot(!(zero == 0.0f))) {
        const int64_t k = k0 + (lane & 31);
        const double xk = snk[3 * k], yk = snk[3 * k + 1], zk = snk[3 * k + 2];
        const float nx = snk_n[3 * k], ny = snk_n[3 * k + 1], nz = snk_n[3 * k + 2];
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int j = 0; j < 16; ++j)
                re[c][j] = im[c][j] = 0.0f;
#pragma unroll 1
        for (int64_t s0 = 0; s0 < S; s0 += 2) {
            const float2 w = Wf[(s0 + half) * GW_B + col];
            const float *q = src + 3 * (s0 + half);
            const GwPair g =
                gw_pair<LOSSY>(q[0], q[1], q[2], xk, yk, zk, nx, ny, nz, ex, ey, ez, kw, alpha);
            const float p[3] = {g.px, g.py, g.pz};
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const float gr = g.Lr * p[c], gi = g.Li * p[c];
                re[c] = __builtin_amdgcn_mfma_f32_32x32x2f32(gr, w.x, re[c], 0, 0, 0);
                re[c] = __builtin_amdgcn_mfma_f32_32x32x2f32(-gi, w.y, re[c], 0, 0, 0);
                im[c] = __builtin_amdgcn_mfma_f32_32x32x2f32(gr, w.y, im[c], 0, 0, 0);
                im[c] = __builtin_amdgcn_mfma_f32_32x32x2f32(gi, w.x, im[c], 0, 0, 0);
            }
        }
    }
    // D[i][j]: lane holds column j = lane % 32, register r holds row
    //     i = 8*(r/4) + 4*(lane/32) + r%4
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int i = 8 * (r >> 2) + 4 * half + (r & 3);
            out[((f * 3 + c) * K + k0 + i) * GW_B + col] = make_float2(re[c][r], im[c][r]);
        }
}

// Large problems: a workgroup owns 64 sinks x 64 sets at one frequency.  Four
// wavefronts (one a SIMD) only multiply -- 32 x 32 x 3 components each -- and four
// only prepare the next step's operands in LDS: G for 64 sinks x 16 sources, 4
// pairs a lane, and the weights, both already split.  72 matrix instructions
// (2,304 cycles) then stand beside about 500 vector instructions of the SIMD's
// other wavefront, and neither waits for the other but at one barrier a step.
template <bool LOSSY>
__global__ __launch_bounds__(512, 2) void k_gw_tile(
    const float *__restrict__ src, int64_t S, const float *__restrict__ snk,
    const float *__restrict__ snk_n, int64_t K, float ex, float ey, float ez,
    const double *__restrict__ kf, double alpha, const float2 *__restrict__ W,
    float2 *__restrict__ out)
{
    // [buffer][plane][half-wave's k][row or set] x 8 bfloat16
    __shared__ __align__(16) char s_g[2][GW_PLANES * 2048];
    __shared__ __align__(16) char s_w[2][6 * 2048];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t f = blockIdx.y;
    const int64_t k0 = (int64_t)blockIdx.x * 64;
    const double kw = kf[f];
    const float2 *Wf = W + f * S * GW_B;
    const int64_t steps = S / GW_KC;
    if (wave >= 4) {
        // operands: sink (and set) `lane`, sources 4 q .. 4 q + 3 of the step
        const int q4 = wave - 4;
        const int64_t k = k0 + lane < K ? k0 + lane : K - 1;
        const double xk = snk[3 * k], yk = snk[3 * k + 1], zk = snk[3 * k + 2];
        const float nx = snk_n[3 * k], ny = snk_n[3 * k + 1], nz = snk_n[3 * k + 2];
        const int at = (q4 >> 1) * 1024 + lane * 16 + (q4 & 1) * 8;
        float pos[12];
        float2 w[4];
        auto load = [&](int64_t t) {
            const int64_t s = (t < steps ? t : 0) * GW_KC + 4 * q4;
#pragma unroll
            for (int i = 0; i < 12; ++i)
                pos[i] = src[3 * s + i];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                w[i] = Wf[(s + i) * GW_B + lane];
        };
        auto generate = [&](char *gb, char *wb) {
            uint2 h[3];
            uint2 *qw = reinterpret_cast<uint2 *>(wb + at);
            split3(w[0].x, w[1].x, h[0].x, h[1].x, h[2].x);
            split3(w[2].x, w[3].x, h[0].y, h[1].y, h[2].y);
#pragma unroll
            for (int i = 0; i < 3; ++i)
                qw[i * 256] = h[i];
            split3(w[0].y, w[1].y, h[0].x, h[1].x, h[2].x);
            split3(w[2].y, w[3].y, h[0].y, h[1].y, h[2].y);
#pragma unroll
            for (int i = 0; i < 3; ++i)
                qw[(3 + i) * 256] = h[i];
            float Lr[4], Li[4], p[3][4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const GwPair g = gw_pair<LOSSY>(pos[3 * i], pos[3 * i + 1], pos[3 * i + 2], xk, yk, zk,
                                                nx, ny, nz, ex, ey, ez, kw, alpha);
                Lr[i] = g.Lr; Li[i] = g.Li;
                p[0][i] = g.px; p[1][i] = g.py; p[2][i] = g.pz;
            }
            uint2 *q = reinterpret_cast<uint2 *>(gb + at);
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                split3(Lr[0] * p[c][0], Lr[1] * p[c][1], h[0].x, h[1].x, h[2].x);
                split3(Lr[2] * p[c][2], Lr[3] * p[c][3], h[0].y, h[1].y, h[2].y);
#pragma unroll
                for (int i = 0; i < 3; ++i)
                    q[(6 * c + i) * 256] = h[i];
                split3(Li[0] * p[c][0], Li[1] * p[c][1], h[0].x, h[1].x, h[2].x);
                split3(Li[2] * p[c][2], Li[3] * p[c][3], h[0].y, h[1].y, h[2].y);
#pragma unroll
                for (int i = 0; i < 3; ++i)
                    q[(6 * c + 3 + i) * 256] = h[i];
            }
        };
        load(0);
        generate(s_g[0], s_w[0]);
        load(1);
        __syncthreads();
        for (int64_t t = 0; t < steps; ++t) {
            if (t + 1 < steps) {
                generate(s_g[(t + 1) & 1], s_w[(t + 1) & 1]);
                load(t + 2);
            }
            __syncthreads();
        }
        return;
    }
    const int rt = wave >> 1, ct = wave & 1;
    const int arow = (lane >> 5) * 1024 + (rt * 32 + (lane & 31)) * 16;
    const int bcol = (lane >> 5) * 1024 + (ct * 32 + (lane & 31)) * 16;
    f32x16 re[3] = {}, im[3] = {};
    Planes gr, gi, wr, wi, nwi;
    auto read_g = [&](Planes &a, Planes &b, const char *g, int c) {
#pragma unroll
        for (int h = 0; h < 3; ++h) {
            a.h[h] = *reinterpret_cast<const bf16x8 *>(g + arow + (6 * c + h) * 2048);
            b.h[h] = *reinterpret_cast<const bf16x8 *>(g + arow + (6 * c + 3 + h) * 2048);
        }
    };
    auto read_w = [&](Planes &a, Planes &b, const char *w) {
#pragma unroll
        for (int h = 0; h < 3; ++h) {
            a.h[h] = *reinterpret_cast<const bf16x8 *>(w + bcol + h * 2048);
            b.h[h] = *reinterpret_cast<const bf16x8 *>(w + bcol + (3 + h) * 2048);
        }
    };
    __builtin_amdgcn_s_setprio(2);
    __syncthreads();
    read_w(wr, wi, s_w[0]);
    read_g(gr, gi, s_g[0], 0);
    for (int64_t t = 0; t < steps; ++t) {
        const char *g = s_g[t & 1];
#pragma unroll
        for (int h = 0; h < 3; ++h)
            nwi.h[h] = flipped(wi.h[h]);
        Planes ar, ai;
        f32x16 r, i;
        read_g(ar, ai, g, 1);
        gw_products(gr, gi, wr, wi, nwi, r, i);
        re[0] += r;
        im[0] += i;
        read_g(gr, gi, g, 2);
        gw_products(ar, ai, wr, wi, nwi, r, i);
        re[1] += r;
        im[1] += i;
        // every read of this buffer is done: the next step's operands are there
        __syncthreads();
        Planes nr, ni;
        read_w(nr, ni, s_w[(t + 1) & 1]);
        read_g(ar, ai, s_g[(t + 1) & 1], 0);
        gw_products(gr, gi, wr, wi, nwi, r, i);
        re[2] += r;
        im[2] += i;
        wr = nr;
        wi = ni;
        gr = ar;
        gi = ai;
    }
    if (k0 + 32 * rt < K)
        gw_finish<LOSSY>(re, im, src, S, snk, snk_n, K, k0 + 32 * rt, ex, ey, ez, kw, alpha, Wf, out,
                         32 * ct + (lane & 31), f);
}

// Small problems: a workgroup owns 32 sinks x 32 sets, and its nw wavefronts split
// the sources, so that few tiles still fill the chip.  A lane prepares its own
// share of the A operand (sink lane % 32, sources 8 (lane / 32) .. + 7 of the
// step) and of the weights in registers: nothing is shared and nothing waits
// until the wavefronts' sums are added, two by two in a fixed order.
template <bool LOSSY>
__global__ __launch_bounds__(64 * GW_MAX_WAVES, 2) void k_gw_mfma(
    const float *__restrict__ src, int64_t S, const float *__restrict__ snk,
    const float *__restrict__ snk_n, int64_t K, float ex, float ey, float ez,
    const double *__restrict__ kf, double alpha, const float2 *__restrict__ W,
    float2 *__restrict__ out)
{
    extern __shared__ float s_part[];  // nw / 2 wavefronts' sums
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const int half = lane >> 5;
    const int64_t f = blockIdx.y;
    const int64_t k0 = (int64_t)(blockIdx.x >> 1) * GW_M;
    const int64_t k = k0 + (lane & 31);
    const int col = (blockIdx.x & 1) * GW_N + (lane & 31);
    const double kw = kf[f];
    const double xk = snk[3 * k], yk = snk[3 * k + 1], zk = snk[3 * k + 2];
    const float nx = snk_n[3 * k], ny = snk_n[3 * k + 1], nz = snk_n[3 * k + 2];
    const float2 *Wf = W + f * S * GW_B;
    f32x16 re[3] = {}, im[3] = {};
    for (int64_t s0 = (int64_t)wave * GW_KC; s0 < S; s0 += (int64_t)nw * GW_KC) {
        const int64_t s = s0 + 8 * half;
        const float2 *q = Wf + s * GW_B + col;
        Planes wr, wi, nwi;
        {
            u32x4 a[3], b[3];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float2 w0 = q[2 * i * GW_B], w1 = q[(2 * i + 1) * GW_B];
                uint32_t q0, q1, q2;
                split3(w0.x, w1.x, q0, q1, q2);
                a[0][i] = q0; a[1][i] = q1; a[2][i] = q2;
                split3(w0.y, w1.y, q0, q1, q2);
                b[0][i] = q0; b[1][i] = q1; b[2][i] = q2;
            }
#pragma unroll
            for (int h = 0; h < 3; ++h) {
                wr.h[h] = __builtin_bit_cast(bf16x8, a[h]);
                wi.h[h] = __builtin_bit_cast(bf16x8, b[h]);
                nwi.h[h] = flipped(wi.h[h]);
            }
        }
        float Lr[8], Li[8], p[3][8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float *x = src + 3 * (s + i);
            const GwPair g = gw_pair<LOSSY>(x[0], x[1], x[2], xk, yk, zk, nx, ny, nz, ex, ey, ez, kw,
                                            alpha);
            Lr[i] = g.Lr; Li[i] = g.Li;
            p[0][i] = g.px; p[1][i] = g.py; p[2][i] = g.pz;
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            u32x4 a[3], b[3];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                uint32_t q0, q1, q2;
                split3(Lr[2 * i] * p[c][2 * i], Lr[2 * i + 1] * p[c][2 * i + 1], q0, q1, q2);
                a[0][i] = q0; a[1][i] = q1; a[2][i] = q2;
                split3(Li[2 * i] * p[c][2 * i], Li[2 * i + 1] * p[c][2 * i + 1], q0, q1, q2);
                b[0][i] = q0; b[1][i] = q1; b[2][i] = q2;
            }
            Planes gr, gi;
#pragma unroll
            for (int h = 0; h < 3; ++h) {
                gr.h[h] = __builtin_bit_cast(bf16x8, a[h]);
                gi.h[h] = __builtin_bit_cast(bf16x8, b[h]);
            }
            f32x16 r, i;
            gw_products(gr, gi, wr, wi, nwi, r, i);
            re[c] += r;
            im[c] += i;
        }
    }
    for (int off = nw >> 1; off > 0; off >>= 1) {
        if (wave >= off && wave < 2 * off) {
            float *q = s_part + (wave - off) * 96 * 64 + lane;
#pragma unroll
            for (int c = 0; c < 3; ++c)
#pragma unroll
                for (int j = 0; j < 16; ++j) {
                    q[(32 * c + j) * 64] = re[c][j];
                    q[(32 * c + 16 + j) * 64] = im[c][j];
                }
        }
        __syncthreads();
        if (wave < off) {
            const float *q = s_part + wave * 96 * 64 + lane;
#pragma unroll
            for (int c = 0; c < 3; ++c)
#pragma unroll
                for (int j = 0; j < 16; ++j) {
                    re[c][j] += q[(32 * c + j) * 64];
                    im[c][j] += q[(32 * c + 16 + j) * 64];
                }
        }
        __syncthreads();
    }
    if (wave == 0)
        gw_finish<LOSSY>(re, im, src, S, snk, snk_n, K, k0, ex, ey, ez, kw, alpha, Wf, out, col, f);
}

// How many wavefronts split the sources (0: k_gw_tile), from what each took in
// units of 0.1 us: a step of k_gw_tile's workgroup, one a CU, 21; a step of a
// k_gw_mfma wavefront 38 alone on its SIMD, 52 beside a second one; adding the
// sums about two steps a level.  Measured (k_gw_tile / k_gw_mfma, us): 1,024
// sources x 2,720 sinks 134 / 74, 4,096 x 2,720 447 / 199, 2,304 x 5,600 x 3
// frequencies 592 / 524; 4,096 x 16,384 593 / 755, 4,096 x 11,328 x 3 1,591 / 1,622,
// 4,096 x 16,384 x 16 9,038 / 11,357.
inline int gw_waves(int64_t K, int64_t F, int64_t steps)
{
    const int64_t tiles = K / GW_M * 2 * F;
    int best = 0;
    int64_t best_cost = ceil_div(ceil_div(K, 64) * F, 256) * (steps + 1) * 21;
    for (int nw = 1, level = 0; nw <= GW_MAX_WAVES && nw <= steps; nw *= 2, ++level) {
        const int64_t a_simd = ceil_div(tiles * nw, 1024);
        const int64_t cost =
            (a_simd == 1 ? 38 : 26 * a_simd) * (ceil_div(steps, nw) + 1 + 2 * level);
        if (cost < best_cost) {
            best = nw;
            best_cost = cost;
        }
    }
    return best;
}

}  // namespace lem

using namespace lem;

extern "C" int lem_gw_mfma(const float *src, int64_t S, float pol_x, float pol_y, float pol_z,
                           const float *snk, const float *snk_n, int64_t K,
                           const double *wavenumbers, int64_t F, double alpha, const float *W,
                           int64_t B, float *out, void *stream)
{
    clear_error();
    LEM_REQUIRE(S > 0 && K > 0 && F > 0, "lem_gw_mfma: empty problem");
    LEM_REQUIRE(src && snk && snk_n && wavenumbers && W && out, "lem_gw_mfma: null pointer");
    LEM_REQUIRE(B == GW_B, "lem_gw_mfma: B must be 64 weight sets");
    LEM_REQUIRE(S % 32 == 0, "lem_gw_mfma: S must be a multiple of 32 (pad with zero weights)");
    LEM_REQUIRE(K % GW_M == 0, "lem_gw_mfma: K must be a multiple of 32 (pad the sinks)");
    LEM_REQUIRE(F <= 65535 && K / GW_M <= 2147483647LL, "lem_gw_mfma: grid too large");
    const float2 *W2 = reinterpret_cast<const float2 *>(W);
    float2 *out2 = reinterpret_cast<float2 *>(out);
    const int nw = gw_waves(K, F, S / GW_KC);
    hipStream_t st = as_stream(stream);
#define LEM_GW(KERNEL, TILE, THREADS, LDS)                                                    \
    do {                                                                                      \
        dim3 grid((unsigned)ceil_div(K, TILE), (unsigned)F);                                  \
        if (alpha != 0.0)                                                                     \
            hipLaunchKernelGGL(KERNEL<true>, grid, dim3(THREADS), LDS, st, src, S, snk, snk_n, K, \
                               pol_x, pol_y, pol_z, wavenumbers, alpha, W2, out2);     \
        else                                                                                  \
            hipLaunchKernelGGL(KERNEL<false>, grid, dim3(THREADS), LDS, st, src, S, snk, snk_n, K, \
                               pol_x, pol_y, pol_z, wavenumbers, alpha, W2, out2);     \
    } while (0)
    if (nw)
        LEM_GW(k_gw_mfma, GW_M / 2, 64 * nw, nw / 2 * 96 * 64 * 4);
    else
        LEM_GW(k_gw_tile, 64, 512, 0);
#undef LEM_GW
    return check_launch("k_gw_mfma");
}
