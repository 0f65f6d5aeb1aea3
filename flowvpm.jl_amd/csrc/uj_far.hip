// uj_far.hip -- the far field of the F32C all-pairs U/J on the matrix cores.
//
// Past the far radius a pair (t, s) has F' = r^-3 and H'' = r^-5, and with
// d = t - s every sum of the U/J kernel (p2p_pair.h, accum_pair) is a
// polynomial in t whose coefficients are sums over the sources of r^-5 times
// a polynomial in s.  With H = r^-5, v = s x Gamma', and positions relative
// to an origin near the targets:
//     A = sum H Gamma'   B_ab = sum H s_a Gamma'_b   C = sum H s^2 Gamma'
//     D_ab = sum H v_a s_b   E = sum H s^2 v         (27 sums per target)
//     W'  = t^2 A - 2 t_a B_a + C                 (r^2 = t^2 - 2 t.s + s^2)
//     U'  = t x W' - (t^2 V - 2 D t + E),         V = sum H v (from B)
//     Jhv = (t x A) t^T - t x B_b - V t^T + D.
// So a (target, source) block is a matrix product: the H of its pairs times
// the 27 columns of its sources.  The VALU kernel spends 33 instructions per
// pair; here the VALU only turns r^2 into H (rsq, two products, and the two
// FP16 halves), and the matrix cores do both contractions.
//
//  * r^2 of 32 sources x 32 targets is one 32x32x16 product of -2 s.t and t^2,
//    with s, t and t^2 split into two FP16 parts each, onto s^2 in FP32 as the
//    accumulator's start: the unit cuts each of 8 products at 2^-24 of the
//    largest, and s^2 among them would cut the others always toward r^2 = s^2.
//  * H = h1 + h2 and column = c1 + c2 in FP16 parts (22 bits, of H below 1/4
//    down to 20, where h2 is subnormal), h1 c1 + h1 c2 + h2 c1 in FP32
//    accumulators: three 32x32x16 products per 16 sources.  The r^2 product
//    leaves a lane with its target's H in exactly the register order the
//    second product reads as its left operand (the sources in permuted order,
//    which the columns' rows follow), so nothing moves between lanes.
//  * Scales: positions are divided by R = 2^k >= every |s| and |t| of the
//    (target block, 256-source tile), strengths by the tile's largest
//    component (a power of two).  A wave of 64 targets takes a group of 64
//    sources here when the gap between their boxes is at least the group's
//    far radius, the wave's reach from the origin (then |t| <= r, |s| <= 2 r:
//    the terms of r^2 reach 9 r^2, three bits, those of U 27 r^3, five), and
//    R / 8 (then H <= 2^15 fits FP16, and r <= 2 R keeps H >= 1/32).  The rest
//    goes to uj_rest_kernel, the VALU pair code: the bits of one word per
//    (block, tile), computed once, tell both kernels who takes which group.
//  * The FP32 accumulators are added to FP64 sums after every 128 sources; the
//    polynomials in t are formed once per target in FP64.
//  * What is the same for every source does not average out: v_rsq_f32's mean
//    error (kRsqMean) and the target's rounding (move_u) are taken out of the
//    sums.
// Error against 64 bits per unit of the summation scale (RMS over targets), all
// pairs in FP32 -> here: U of the 2^20 jet 1.3e-8 -> 5.4e-9, of the 65,536
// leapfrog rings 1.65e-8 -> 1.1e-8 and cloud 1.88e-9 -> 1.86e-9, J 3.8e-8 ->
// 1.6e-8, 7.7e-8 -> 3.0e-8 and 8.2e-9 -> 5.5e-9 (the rest kernel's shorter
// chains).  With s^2 among the products, a fold per 256 sources and both means
// left in, U was 2.4e-8, 1.7e-8 and 1.9e-9, and the jet took 337 ms instead of
// 353 (s^2 from LDS 8 ms, the second fold 9).
// Measured: U/J of the 2^20 jet 709 -> 353 ms (1.55e12 -> 3.1e12 pairs/s), of
// the 65,536 cloud 3.72 -> 2.50 ms and of the leapfrog rings 3.26 -> 1.80 ms.
// The far kernel is bound by the VALU: per pair one rsq (8.3 cycles of a SIMD
// for 64 pairs), three products (2.6 each), two packed conversions of two (4.6)
// and a fma_mix (4.4) are 25 of the 43 cycles that it takes, at 2.1 GHz; the
// matrix products keep their unit busy a third of the time beside them.
#include <algorithm>
#include <cfloat>

#include "p2p_pair.h"
#include "uj_far.h"

namespace vpm {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kCols = 27;            // columns of a source
constexpr int kColLd = kTile + 8;    // halves per column row in LDS: 33 x 16 bytes, so 16 rows cover all banks
constexpr int kColShift = 13;        // columns are scaled by 2^13
constexpr float kLowScale = 64.f;    // scale of the low FP16 part of a position
constexpr float kSqScale = 4096.f;   // scale of t^2 in the r^2 product
// v_rsq_f32 is low by 5.8e-9 of its result on [1, 2) and 8.1e-9 on [2, 4)
// (means weighted by 1/x), so r^-5 by 3.5e-8 wherever r lies.
constexpr double kRsqMean = 1.0 + 3.5e-8;
// The far kernel pays from 16,384 particles.  U/J of the cloud, the jet, the
// leapfrog rings and a thin ring with every pair on the VALU, and with it: 0.208
// / 0.233, 0.183 / 0.194, 0.223 / 0.259 and 0.182 / 0.198 ms at 12,288 (boxes
// of 64 particles are too large for most pairs to be far), 0.320 / 0.322, 0.291
// / 0.301, 0.347 / 0.318 and 0.278 / 0.274 at 16,384, 0.457 / 0.404, 0.415 /
// 0.355, 0.459 / 0.423 and 0.396 / 0.344 at 20,000.  Where nearly every pair is
// near it costs the words and the smaller tiles of the rest kernel: the 65,536
// cloud with four times its core sizes 6.5 -> 6.9 ms, ten times 6.9 -> 7.2, one
// of density ~ r^-2 3.8 -> 4.1 (0.38 -> 0.41 at 16,384, 18.3 -> 14.3 at 150,000).
constexpr int64_t kFarPairs = (int64_t)1 << 28;
constexpr int64_t kFarMin = 2048;
constexpr int kFarThreads = 512;     // threads of a block of 256 targets

// Box of each run of 64 consecutive particles: lo, hi, then the largest
// far-field r^2 threshold and the largest |Gamma'| component (cut != null).
__global__ __launch_bounds__(kBlock) void far_box_kernel(const double* __restrict__ pos, int64_t ld, int64_t t0,
                                                         int64_t n, const float* __restrict__ cut,
                                                         const float4* __restrict__ gs, double* __restrict__ box)
{
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    const int64_t grp = i >> 6;
    if (grp * 64 >= n) return;   // whole waves
    const int64_t k = t0 + min(i, n - 1);
    const WaveBox64 b = wave_box64(pos[k], pos[ld + k], pos[2 * ld + k]);
    float c = 0.f, g = 0.f;
    if (cut) {
        const float4 q = gs[k];
        c = cut[k];
        g = fmaxf(fabsf(q.x), fmaxf(fabsf(q.y), fabsf(q.z)));
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            c = fmaxf(c, __shfl_xor(c, off));
            g = fmaxf(g, __shfl_xor(g, off));
        }
    }
    if ((threadIdx.x & 63) == 0) {
        double* o = box + 8 * grp;
        for (int a = 0; a < 3; ++a) { o[a] = b.lo[a]; o[3 + a] = b.hi[a]; }
        o[6] = c;
        o[7] = g;
    }
}

// Origin of a target block: the centre of the box of its waves' boxes.
__device__ __forceinline__ void block_origin(const double* __restrict__ tbox, int64_t w0, int64_t w1, double (&O)[3],
                                             double (&half)[3])
{
    for (int a = 0; a < 3; ++a) {
        double lo = tbox[8 * w0 + a], hi = tbox[8 * w0 + 3 + a];
        for (int64_t w = w0 + 1; w < w1; ++w) {
            lo = fmin(lo, tbox[8 * w + a]);
            hi = fmax(hi, tbox[8 * w + 3 + a]);
        }
        O[a] = 0.5 * (lo + hi);
        half[a] = 0.5 * (hi - lo);
    }
}

// One word per (block of 4 target waves, tile of 4 source groups): bit 4 w +
// g set when wave w takes group g in the far kernel, bits 16-23 k + 64, bits
// 24-31 the exponent of the tile's strengths + 128.  Waves and groups past
// the end have their bit set (nothing is left for the VALU kernel).
__global__ __launch_bounds__(kBlock) void far_word_kernel(const double* __restrict__ tbox, int64_t nwave,
                                                          const double* __restrict__ gbox, int64_t ngroup,
                                                          int64_t ntile, uint32_t* __restrict__ words)
{
    const int64_t tile = (int64_t)blockIdx.y * kBlock + threadIdx.x;
    if (tile >= ntile) return;
    const int64_t w0 = (int64_t)blockIdx.x * 4, w1 = min(w0 + 4, nwave);
    const int64_t g0 = tile * 4, g1 = min(g0 + 4, ngroup);
    double O[3], half[3];
    block_origin(tbox, w0, w1, O, half);
    double r2 = half[0] * half[0] + half[1] * half[1] + half[2] * half[2];
    double gm = 0.0;
    for (int64_t g = g0; g < g1; ++g) {
        const double* G = gbox + 8 * g;
        double s2 = 0.0;
        for (int a = 0; a < 3; ++a) {
            const double e = fmax(fabs(G[a] - O[a]), fabs(G[3 + a] - O[a]));
            s2 = fma(e, e, s2);
        }
        r2 = fmax(r2, s2);
        gm = fmax(gm, G[7]);
    }
    int k = 0, ge = 0;
    (void)frexp(sqrt(r2) * (1.0 + 1e-6), &k);   // 2^k > every |s|, |t|
    if (gm > 0.0) (void)frexp(gm * (1.0 + 1e-6), &ge);
    // scales and their products stay well inside FP32 (frexp gives an
    // infinity, a strength beyond FP32 or a distance squared, the exponent 0)
    const bool ok = r2 < INFINITY && gm < INFINITY && k >= -24 && k <= 24 && ge >= -100 && ge <= 60 && ge - 5 * k <= 100;
    const double rmin2 = ldexp(1.0, 2 * k - 6) * (1.0 + 1e-4);
    uint32_t bits = 0;
    for (int w = 0; w < 4; ++w) {
        if (w0 + w >= w1) { bits |= 15u << (4 * w); continue; }
        const double* T = tbox + 8 * (w0 + w);
        double reach2 = 0.0;
        for (int a = 0; a < 3; ++a) {
            const double e = fmax(fabs(T[a] - O[a]), fabs(T[3 + a] - O[a]));
            reach2 = fma(e, e, reach2);
        }
        for (int g = 0; g < 4; ++g) {
            if (g0 + g >= g1) { bits |= 1u << (4 * w + g); continue; }
            const double* G = gbox + 8 * (g0 + g);
            double gap2 = 0.0;
            for (int a = 0; a < 3; ++a) {
                const double e = fmax(fmax(G[a] - T[3 + a], T[a] - G[3 + a]), 0.0);
                gap2 = fma(e, e, gap2);
            }
            if (ok && gap2 >= fmax(fmax(G[6] * (1.0 + 1e-4), reach2), rmin2)) bits |= 1u << (4 * w + g);
        }
    }
    words[(int64_t)blockIdx.x * ntile + tile] = bits | ((uint32_t)(k + 64) & 255u) << 16 | (uint32_t)(ge + 128) << 24;
}

__device__ __forceinline__ void split16(double x, _Float16& h, _Float16& l)
{
    h = (_Float16)(float)x;
    l = (_Float16)(float)(x - (double)(float)h);
}

__device__ __forceinline__ double square3(const float (&x)[3])
{
    return fma((double)x[2], (double)x[2], fma((double)x[1], (double)x[1], (double)x[0] * x[0]));
}

// x = h + l / kLowScale; returns the represented value
__device__ __forceinline__ float split_pos(float x, _Float16& h, _Float16& l)
{
    h = (_Float16)x;
    l = (_Float16)((x - (float)h) * kLowScale);
    return fmaf((float)l, 1.f / kLowScale, (float)h);
}

__device__ __forceinline__ floatx16 mfma16(half8 a, half8 b, floatx16 c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// U of the 14 sums moved by d, to first order (J as in add_f32c_to_record).
__device__ __forceinline__ void move_u(const double (&d)[3], double (&a)[kAccF32])
{
    const double u0 = -3.0 * (a[6] * d[0] + a[9] * d[1] + a[12] * d[2]) + a[5] * d[1] - a[4] * d[2];
    const double u1 = -3.0 * (a[7] * d[0] + a[10] * d[1] + a[13] * d[2]) - a[5] * d[0] + a[3] * d[2];
    const double u2 = -3.0 * (a[8] * d[0] + a[11] * d[1] - (a[6] + a[10]) * d[2]) + a[4] * d[0] - a[3] * d[1];
    a[0] += u0;
    a[1] += u1;
    a[2] += u2;
}

// The 14 sums of accum_pair from the 27 basis sums S of a target at t.
__device__ __forceinline__ void far_combine(const double (&t)[3], const double* S, double (&out)[kAccF32])
{
    const double* A = S;
    const double* B = S + 3;      // B[3 a + b] = sum H s_a Gamma_b
    const double* Cc = S + 12;
    const double* D = S + 15;     // D[3 a + b] = sum H v_a s_b
    const double* E = S + 24;
    const double t2 = t[0] * t[0] + t[1] * t[1] + t[2] * t[2];
    const double V[3] = {B[5] - B[7], B[6] - B[2], B[1] - B[3]};
    double W[3], FV[3];
#pragma unroll
    for (int b = 0; b < 3; ++b) {
        W[b] = t2 * A[b] - 2.0 * (t[0] * B[b] + t[1] * B[3 + b] + t[2] * B[6 + b]) + Cc[b];
        FV[b] = t2 * V[b] - 2.0 * (D[3 * b] * t[0] + D[3 * b + 1] * t[1] + D[3 * b + 2] * t[2]) + E[b];
    }
    out[0] = t[1] * W[2] - t[2] * W[1] - FV[0];
    out[1] = t[2] * W[0] - t[0] * W[2] - FV[1];
    out[2] = t[0] * W[1] - t[1] * W[0] - FV[2];
    out[3] = W[0];
    out[4] = W[1];
    out[5] = W[2];
    const double tA[3] = {t[1] * A[2] - t[2] * A[1], t[2] * A[0] - t[0] * A[2], t[0] * A[1] - t[1] * A[0]};
#pragma unroll
    for (int b = 0; b < 3; ++b) {
        const double* Bb = B + 3 * b;   // sum H s_b Gamma
        const double tB[3] = {t[1] * Bb[2] - t[2] * Bb[1], t[2] * Bb[0] - t[0] * Bb[2], t[0] * Bb[1] - t[1] * Bb[0]};
#pragma unroll
        for (int a = 0; a < 3; ++a)
            if (3 * b + a < 8) out[6 + 3 * b + a] = (tA[a] - V[a]) * t[b] - tB[a] + D[3 * a + b];
    }
}

// H of 8 pairs of one target as FP16 parts, from r^2 (scaled)
__device__ __forceinline__ void weights(const float* r2, half8& h1, half8& h2)
{
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
        float H[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float ri = rsq(r2[i + e]);
            const float ri2 = ri * ri;
            H[e] = ri2 * ri2 * ri;
        }
        // remainders by v_fma_mix_f32 (one instruction instead of an unpack
        // and a subtraction), both halves by packed conversions
        const half2v hp = {(_Float16)H[0], (_Float16)H[1]};
        float l0, l1;
        asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel_hi:[0,0,1]" : "=v"(l0) : "v"(H[0]), "v"(hp));
        asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "=v"(l1) : "v"(H[1]), "v"(hp));
        const half2v lp = {(_Float16)l0, (_Float16)l1};
        h1[i] = hp[0];
        h1[i + 1] = hp[1];
        h2[i] = lp[0];
        h2[i + 1] = lp[1];
    }
}

// 8 waves of 32 targets (two waves to a word's 64), 256 sources per tile.
// Four waves per SIMD: a wave issues at most every ~5 cycles, a single-rate
// instruction takes 2.6.
__global__ __launch_bounds__(kFarThreads, 4) void uj_far_kernel(
    const double* __restrict__ tpos, int64_t tld, int64_t t0, int64_t nt, const double* __restrict__ tbox,
    const double* __restrict__ spos, int64_t sld, const float4* __restrict__ sgs, int64_t ns,
    const uint32_t* __restrict__ words, int64_t ntile, int64_t chunk, double* __restrict__ part, int64_t pld)
{
    // columns [part][column][source], the sources' halves of the r^2 product
    // and their s^2; the basis sums at the end reuse the space, four waves at a time
    constexpr int kColBytes = 2 * kCols * kColLd * 2;
    constexpr int kSumLd = kCols + 1;
    constexpr int kSumBytes = 4 * 32 * kSumLd * 8;
    constexpr int kStageBytes = kColBytes + 2 * kTile * 16 + kTile * 4;
    __shared__ __attribute__((aligned(16))) char smem[kStageBytes > kSumBytes ? kStageBytes : kSumBytes];
    _Float16* lcol = (_Float16*)smem;
    half8* lr = (half8*)(smem + kColBytes);
    float* ls2 = (float*)(smem + kColBytes + 2 * kTile * 16);

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = lane & 31, hh = lane >> 5;
    const int64_t blk = blockIdx.x;
    const int64_t i0 = blk * kBlock + wave * 32;
    const int64_t nwave = (nt + 63) / 64;
    double O[3], half_[3];
    block_origin(tbox, blk * 4, min(blk * 4 + 4, nwave), O, half_);
    float tf[3];
    {
        const int64_t k = t0 + min(i0 + m, nt - 1);
        for (int a = 0; a < 3; ++a) tf[a] = (float)(tpos[a * tld + k] - O[a]);
    }
    const int n = min(m, kCols - 1);
    const int deg = n < 3 ? 0 : n < 12 ? 1 : n < 24 ? 2 : 3;
    // staging: threads 0-255 and 256-511 share the columns of source `src`
    const int src = tid & (kTile - 1);
    const int p = (src & ~12) | ((src & 4) << 1) | ((src & 8) >> 1);   // the source's place in its columns

    const floatx16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    floatx16 acc = zero;
    double sum[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) sum[i] = 0.0;
    half8 T;
    float trep[3] = {0.f, 0.f, 0.f};   // the target as T has it (the same in every scale)
    int kcur = 1000;

    const int64_t c0 = (int64_t)blockIdx.y * chunk, c1 = min(c0 + chunk, ntile);
    for (int64_t tile = c0; tile < c1; ++tile) {
        const uint32_t word = words[blk * ntile + tile];
        if ((word & 0xffffu) == 0) continue;
        const int k = (int)(word >> 16 & 255u) - 64, ge = (int)(word >> 24) - 128;
        __syncthreads();   // the previous tile's readers are done
        {
            const int64_t j = tile * kTile + src;
            const bool real = j < ns;
            const int64_t jj = real ? j : ns - 1;
            const double inv = ldexp(1.0, -k);
            float s[3];
            for (int a = 0; a < 3; ++a) {
                const float x = (float)((spos[a * sld + jj] - O[a]) * inv);
                s[a] = real ? x : 2.f;   // padding: zero strength, away from every target
            }
            const float4 gq = sgs[jj];
            const float gsc = real ? ldexpf(1.f, kColShift - ge) : 0.f;
            const float g[3] = {gq.x * gsc, gq.y * gsc, gq.z * gsc};
            const auto put = [&](int c, float x, int d, float y) {   // columns c and d
                half2v h = {(_Float16)x, (_Float16)y};
                asm("" : "+v"(h));
                const half2v l = {(_Float16)(x - (float)h[0]), (_Float16)(y - (float)h[1])};
                lcol[c * kColLd + p] = h[0];
                lcol[(kCols + c) * kColLd + p] = l[0];
                if (d != c) {
                    lcol[d * kColLd + p] = h[1];
                    lcol[(kCols + d) * kColLd + p] = l[1];
                }
            };
            if (wave < 4) {
                half8 r0, r1;
                float st[3];
                for (int a = 0; a < 3; ++a) {
                    _Float16 h, l;
                    st[a] = split_pos(s[a], h, l);
                    r0[a] = h;
                    r0[3 + a] = l;
                    r1[a] = (_Float16)((float)h * (1.f / kLowScale));
                    r1[3 + a] = l;
                }
                r0[6] = r0[7] = (_Float16)(1.f / kSqScale);
                r1[6] = r1[7] = (_Float16)0.f;
                ls2[src] = (float)square3(st);
                lr[src] = r0;
                lr[kTile + src] = r1;
                put(0, g[0], 1, g[1]);
                put(2, g[2], 3, s[0] * g[0]);
                put(4, s[0] * g[1], 5, s[0] * g[2]);
                put(6, s[1] * g[0], 7, s[1] * g[1]);
                put(8, s[1] * g[2], 9, s[2] * g[0]);
                put(10, s[2] * g[1], 11, s[2] * g[2]);
            } else {
                const float s2 = fmaf(s[2], s[2], fmaf(s[1], s[1], s[0] * s[0]));
                const float v[3] = {fmaf(s[1], g[2], -s[2] * g[1]), fmaf(s[2], g[0], -s[0] * g[2]),
                                    fmaf(s[0], g[1], -s[1] * g[0])};
                put(12, s2 * g[0], 13, s2 * g[1]);
                put(14, s2 * g[2], 15, v[0] * s[0]);
                put(16, v[0] * s[1], 17, v[0] * s[2]);
                put(18, v[1] * s[0], 19, v[1] * s[1]);
                put(20, v[1] * s[2], 21, v[2] * s[0]);
                put(22, v[2] * s[1], 23, v[2] * s[2]);
                put(24, s2 * v[0], 25, s2 * v[1]);
                put(26, s2 * v[2], 26, s2 * v[2]);
            }
        }
        __syncthreads();
        const uint32_t my = i0 < nt ? (word >> (4 * (wave >> 1))) & 15u : 0u;
        if (!my) continue;
        if (k != kcur) {
            kcur = k;
            const float inv = ldexpf(1.f, -k);
            float st[3];
            for (int a = 0; a < 3; ++a) {
                _Float16 h, l;
                st[a] = split_pos(tf[a] * inv, h, l);
                const float x = -2.f * (hh ? (float)l : (float)h);
                T[a] = (_Float16)x;
                T[3 + a] = (_Float16)(x * (hh ? 1.f / (kLowScale * kLowScale) : 1.f / kLowScale));
            }
            for (int a = 0; a < 3; ++a) trep[a] = ldexpf(st[a], k);
            _Float16 q1, q2;
            split16(square3(st) * kSqScale, q1, q2);
            T[6] = hh ? (_Float16)0.f : q1;
            T[7] = hh ? (_Float16)0.f : q2;
        }
        const double sc = ldexp(kRsqMean, ge - kColShift + k * (deg - 5));
        const auto fold = [&]() {
#pragma unroll
            for (int i = 0; i < 16; ++i) sum[i] = fma((double)acc[i], sc, sum[i]);
            acc = zero;
        };
        for (int g = 0; g < 4; ++g) {
            if (g == 2) fold();
            if (!((my >> g) & 1u) || tile * kTile + g * 64 >= ns) continue;
            const half8* rp = lr + hh * kTile + g * 64 + m;
            const _Float16* cp = lcol + n * kColLd + g * 64 + hh * 8;
            floatx16 ra, rb;   // s^2 of the lane's rows, then r^2
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float* p2 = ls2 + g * 64 + 8 * q + 4 * hh;
                const float4 x = *(const float4*)p2, y = *(const float4*)(p2 + 32);
                ra[4 * q] = x.x; ra[4 * q + 1] = x.y; ra[4 * q + 2] = x.z; ra[4 * q + 3] = x.w;
                rb[4 * q] = y.x; rb[4 * q + 1] = y.y; rb[4 * q + 2] = y.z; rb[4 * q + 3] = y.w;
            }
            ra = mfma16(rp[0], T, ra);
            rb = mfma16(rp[32], T, rb);
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                const floatx16& r2 = ks < 2 ? ra : rb;
                float x[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) x[i] = r2[8 * (ks & 1) + i];
                const half8 b1 = *(const half8*)(cp + ks * 16), b2 = *(const half8*)(cp + kCols * kColLd + ks * 16);
                half8 h1, h2;
                weights(x, h1, h2);
                acc = mfma16(h2, b1, acc);
                acc = mfma16(h1, b2, acc);
                acc = mfma16(h1, b1, acc);
            }
        }
        fold();
    }
    // the wave's 32 targets x 27 sums to LDS, then a target per lane
    for (int half = 0; half < 2; ++half) {
        __syncthreads();
        if ((wave >> 2) != half) continue;
        double* ls = (double*)smem + (wave & 3) * 32 * kSumLd;
        if (m < kCols) {
#pragma unroll
            for (int i = 0; i < 16; ++i) ls[(8 * (i >> 2) + 4 * hh + (i & 3)) * kSumLd + m] = sum[i];
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const int64_t i = i0 + lane;
        if (lane < 32 && i < nt) {
            // sums for the target as the weights had it, then moved to its
            // place: its rounding is the same for every source, and left in
            // the weights it is the largest error of U
            double t[3], d[3], out[kAccF32];
            for (int a = 0; a < 3; ++a) {
                t[a] = trep[a];
                d[a] = tpos[a * tld + t0 + i] - O[a] - t[a];
            }
            far_combine(t, ls + lane * kSumLd, out);
            move_u(d, out);
            double* o = part + (int64_t)blockIdx.y * kAccF32 * pld + i;
#pragma unroll
            for (int c = 0; c < kAccF32; ++c) o[c * pld] = out[c];
        }
    }
}

// The groups the far kernel leaves, on the VALU: each wave of 64 targets
// walks the zero bits of its words by itself (no barrier; block y of gridDim.y
// takes every gridDim.y-th tile, which spreads a wave's near tiles, mostly
// neighbours in the sort order, over the blocks) and stages a group of 64
// sources at a time in its own LDS slot.
template <int K>
__global__ __launch_bounds__(kBlock, 4) void uj_rest_kernel(
    const double* __restrict__ tpos, int64_t tld, int64_t t0, int64_t nt, const double* __restrict__ spos, int64_t sld,
    const float4* __restrict__ sgs, const float* __restrict__ scut, int64_t ns, const uint32_t* __restrict__ words,
    int64_t ntile, double* __restrict__ part, int64_t pld)
{
    __shared__ float4 lpos_all[kBlock / 64][64];   // s'_hi, far-field r^2 threshold
    __shared__ float4 lgs_all[kBlock / 64][64];    // Gamma', 1/sigma
    __shared__ float4 llo_all[kBlock / 64][64];    // s'_lo
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t i0 = (int64_t)blockIdx.x * kBlock + wave * 64;
    if (i0 >= nt) return;   // no block barrier below
    float4* lpos = lpos_all[wave];
    float4* lgs = lgs_all[wave];
    float4* llo = llo_all[wave];
    const int64_t ib = t0 + i0;
    const double ox = tpos[ib], oy = tpos[tld + ib], oz = tpos[2 * tld + ib];
    const bool active = i0 + lane < nt;
    const int64_t it = active ? ib + lane : ib;
    float tx, ty, tz, tlx, tly, tlz;
    split_rel(tpos[it], ox, tx, tlx);
    split_rel(tpos[tld + it], oy, ty, tly);
    split_rel(tpos[2 * tld + it], oz, tz, tlz);
    const WaveBox box = wave_box(tx, ty, tz);

    float sum[kAccF32], err[kAccF32];
#pragma unroll
    for (int c = 0; c < kAccF32; ++c) { sum[c] = 0.f; err[c] = 0.f; }
    const uint32_t* wp = words + (int64_t)blockIdx.x * ntile;
    for (int64_t q = blockIdx.y; q < ntile; q += (int64_t)gridDim.y * 64) {
        const int64_t tl = q + (int64_t)gridDim.y * lane;
        const uint32_t need = tl < ntile ? ~(wp[tl] >> (4 * wave)) & 15u : 0u;
        uint64_t todo = __ballot(need != 0);
        while (todo) {
            const int l = __builtin_ctzll(todo);
            todo &= todo - 1;
            uint32_t bits = __builtin_amdgcn_readlane(need, l);
            const int64_t tile = q + (int64_t)gridDim.y * l;
            while (bits) {
                const int64_t base = tile * kTile + __builtin_ctz(bits) * 64;
                bits &= bits - 1;
                const int n = (int)min((int64_t)64, ns - base);
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                if (lane < n) {
                    const int64_t j = base + lane;
                    float4 p, l4;
                    split_rel(spos[j], ox, p.x, l4.x);
                    split_rel(spos[sld + j], oy, p.y, l4.y);
                    split_rel(spos[2 * sld + j], oz, p.z, l4.z);
                    p.w = scut[j];
                    l4.w = 0.f;
                    lpos[lane] = p;
                    llo[lane] = l4;
                    lgs[lane] = sgs[j];
                }
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                // a fold per group: the groups left here are the near ones,
                // and J loses a digit to FP32 chains over 256 of them
                float acc[kAccF32];
#pragma unroll
                for (int c = 0; c < kAccF32; ++c) acc[c] = 0.f;
                tile_f32c<K, 1, true, false>(n, lpos, lgs, llo, tx, ty, tz, tlx, tly, tlz, box, acc, sum, err);
                fold_twosum(acc, sum, err);
            }
        }
    }
    if (active) {
        double* out = part + (int64_t)blockIdx.y * kAccF32 * pld + i0 + lane;
#pragma unroll
        for (int c = 0; c < kAccF32; ++c) out[c * pld] = (double)sum[c] + (double)err[c];
    }
}

bool far_applies(int kernel, int precision, int64_t nt, int64_t ns)
{
    const bool cheap = kernel == VPM_KERNEL_GAUSSIANERF || kernel == VPM_KERNEL_GAUSSIAN;
    return cheap && precision == VPM_PREC_F32C && nt >= kFarMin && ns >= kFarMin && nt * ns >= kFarPairs;
}

int launch_uj_far(hipStream_t stream, const Staged& T, int64_t t0, int64_t nt, const Staged& S, int64_t ns, int kernel,
                  const FarSplit& k, void* scratch, double* part)
{
    const int64_t nwave = (nt + 63) / 64, ngroup = (ns + 63) / 64;
    const unsigned nblk = (unsigned)((nt + kBlock - 1) / kBlock), ntile = (unsigned)((ns + kTile - 1) / kTile);
    char* p = (char*)scratch;
    double* tbox = (double*)p;
    double* gbox = (double*)(p + far_up256(64 * nwave));
    uint32_t* words = (uint32_t*)(p + far_up256(64 * nwave) + far_up256(64 * ngroup));
    double* rest = part + (size_t)k.far * kAccF32 * (size_t)nt;
    hipLaunchKernelGGL(far_box_kernel, dim3(nblk), dim3(kBlock), 0, stream, T.pos, T.ld, t0, nt, (const float*)nullptr,
                       (const float4*)nullptr, tbox);
    hipLaunchKernelGGL(far_box_kernel, dim3(ntile), dim3(kBlock), 0, stream, S.pos, S.ld, (int64_t)0, ns, S.cut, S.gs,
                       gbox);
    hipLaunchKernelGGL(far_word_kernel, dim3(nblk, (ntile + kBlock - 1) / kBlock), dim3(kBlock), 0, stream,
                       (const double*)tbox, nwave, (const double*)gbox, ngroup, (int64_t)ntile, words);
    hipLaunchKernelGGL(uj_far_kernel, dim3(nblk, (unsigned)k.far), dim3(kFarThreads), 0, stream, T.pos, T.ld, t0, nt,
                       (const double*)tbox, S.pos, S.ld, S.gs, ns, (const uint32_t*)words, (int64_t)ntile, k.chunk,
                       part, nt);
    switch (kernel) {
#define VPM_REST(KID)                                                                                              \
    case KID:                                                                                                      \
        hipLaunchKernelGGL(uj_rest_kernel<KID>, dim3(nblk, (unsigned)k.rest), dim3(kBlock), 0, stream, T.pos, T.ld, \
                           t0, nt, S.pos, S.ld, S.gs, S.cut, ns, (const uint32_t*)words, (int64_t)ntile, rest, nt); \
        break;
        VPM_REST(VPM_KERNEL_GAUSSIAN)
        VPM_REST(VPM_KERNEL_GAUSSIANERF)
#undef VPM_REST
    default:
        return fail(VPM_EINVAL, "unknown kernel id");
    }
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? VPM_OK : hip_fail(e, "uj_far");
}

}  // namespace vpm
