// The feed-forward half of a width-128 block in registers and its weights' way into LDS, shared by the feed-forward kernels
// and the fused column and row blocks (the scheme is described with the kernels).
#pragma once

#include "common.hpp"
#include "device_math.hpp"

namespace tah {

constexpr int CPS = 4;              // 16-column steps (8 KB of a 128-row weight block) per weight slice
constexpr int SLAB = CPS * 8192;    // one weight slice in LDS
constexpr int NSL = 8 * 8192 / SLAB;  // slices per 128 x 128 weight block

// bytes (a multiple of 16 * THREADS) from global to LDS by THREADS threads, 16 bytes a lane; in copy i wavefront w's
// 64 lanes fill the 1 KB at 16 THREADS i + 1024 w (a wavefront-uniform LDS base, the lanes' offsets implicit)
template <int THREADS = 256>
__device__ __forceinline__ void dma_to_lds(const uint8_t *src, uint8_t *dst, int bytes, int tid) {
    for (int o = 0; o < bytes; o += 16 * THREADS)
        __builtin_amdgcn_global_load_lds(src + o + 16 * tid, dst + o + 1024 * (tid >> 6), 16, 0, 0);
}

constexpr int FFW = 4;  // wavefronts (of 32 rows each) per k_ff128 workgroup (eight, one workgroup a CU, measured slower)

// The feed-forward body's start, by all THREADS threads of a workgroup: the first weight slice's copy into slab (two
// slices, 64 KB of LDS) and the first layer's bias into bias1 (256 floats of LDS).
template <int THREADS = 64 * FFW>
__device__ __forceinline__ void ff128_start(uint8_t *slab, float *bias1, const uint8_t *__restrict__ w1img,
                                            const float *__restrict__ b1, int tid) {
    dma_to_lds<THREADS>(w1img, slab, SLAB, tid);
    if (tid < 64) reinterpret_cast<float4 *>(bias1)[tid] = reinterpret_cast<const float4 *>(b1)[tid];
}

// Layer normalisation of this lane's half row xv (columns 16 ks + 8 g + t; the other half on lane l ^ 32) with
// lnw / lnb in place (two passes, biased variance, eps 1e-5), then its split as the B operand of a 128-column product,
// scaled by the row's power of two 2^sx (its largest magnitude below 2^14); returns sx.
__device__ __forceinline__ int norm_split(float (&xv)[8][8], const float *__restrict__ lnw,
                                          const float *__restrict__ lnb, int g, halfx8 (&xh)[8], halfx8 (&xl)[8]) {
    constexpr int E = 128;
    float sum = 0.0f;
#pragma unroll
    for (int ks = 0; ks < 8; ks++)
#pragma unroll
        for (int t = 0; t < 8; t++) sum += xv[ks][t];
    sum = half_sum(sum);
    const float mean = sum / (float)E;
    float sq = 0.0f;
#pragma unroll
    for (int ks = 0; ks < 8; ks++)
#pragma unroll
        for (int t = 0; t < 8; t++) {
            const float dv = xv[ks][t] - mean;
            sq += dv * dv;
        }
    sq = half_sum(sq);
    const float inv = 1.0f / sqrtf(sq / (float)E + 1e-5f);
    float xmax = 0.0f;
#pragma unroll
    for (int ks = 0; ks < 8; ks++) {
        const float4 wa = *reinterpret_cast<const float4 *>(lnw + 16 * ks + 8 * g);
        const float4 wb = *reinterpret_cast<const float4 *>(lnw + 16 * ks + 8 * g + 4);
        const float4 ba = *reinterpret_cast<const float4 *>(lnb + 16 * ks + 8 * g);
        const float4 bb = *reinterpret_cast<const float4 *>(lnb + 16 * ks + 8 * g + 4);
        const float wv[8] = {wa.x, wa.y, wa.z, wa.w, wb.x, wb.y, wb.z, wb.w};
        const float bv[8] = {ba.x, ba.y, ba.z, ba.w, bb.x, bb.y, bb.z, bb.w};
#pragma unroll
        for (int t = 0; t < 8; t++) {
            xv[ks][t] = (xv[ks][t] - mean) * inv * wv[t] + bv[t];
            xmax = fmaxf(xmax, fabsf(xv[ks][t]));
        }
    }
    xmax = half_max(xmax);
    const int sx = shift_for_max(xmax);
#pragma unroll
    for (int ks = 0; ks < 8; ks++) split8(xv[ks], ldexpf(1.0f, sx), xh[ks], xl[ks]);
    return sx;
}

// The next block's key and value projection, formed from a feed-forward's result in the same kernel (ff128_rows with
// KV): img the [2 e][e] weight image (the keys' 128 rows, then the values'), shift its power of two, lnw / lnb the
// next block's first normalisation, b its 2 e biases, out the lane's token's [2 e] row (keys, then values).
struct KvNext {
    const uint8_t *img;
    int shift;
    const float *lnw, *lnb, *b;
    float *out;
};

// x += l2(gelu(l1(norm2 x))) + b2 for 32 rows a wavefront (after ff128_start, all THREADS threads): xv holds this lane's
// half of its row (columns 16 ks + 8 g + t); xrow is the row's storage, which holds x (read back for the residual
// add) and takes the result (not where !live or !keep). With KV the result goes on, still in registers, through kn's
// normalisation and projection (its four weight slices streamed after W2's) to kn.out (not where !live).
template <bool KV = false, int THREADS = 64 * FFW>
__device__ __forceinline__ void ff128_rows(float (&xv)[8][8], bool live, float *xrow, uint8_t *slab, const float *bias1,
                                           const float *__restrict__ lnw, const float *__restrict__ lnb,
                                           const uint8_t *__restrict__ w1img, int s1,
                                           const uint8_t *__restrict__ w2img, const float *__restrict__ b2, int s2,
                                           int tid, const KvNext &kn = KvNext{}, bool keep = true) {
    constexpr int E = 128;
    const int lane = tid & 63;
    const int r32 = lane & 31, g = lane >> 5;
    halfx8 xh[8], xl[8];
    const int sx = norm_split(xv, lnw, lnb, g, xh, xl);

    // H^T = W1 X^T in two halves of 128 hidden units (4 tiles of 32 each); the weights stream as slices of CPS
    // 16-column steps, W1's (half-major) then W2's, slice j into buffer j % 2
    const int arow = sigma32(r32);
    // slices 0 .. 2 NSL - 1: W1 (two 128-row blocks), then 2 NSL .. 4 NSL - 1: W2 (128 rows, 256 columns), then
    // with KV 4 NSL .. 6 NSL - 1: the next block's key and value weights (two 128-row blocks)
    constexpr int NSLICES = (KV ? 6 : 4) * NSL;
    auto slice = [&](int j) {
        return j < 2 * NSL   ? w1img + (size_t)j * SLAB
               : j < 4 * NSL ? w2img + (size_t)(j - 2 * NSL) * SLAB
                             : kn.img + (size_t)(j - 4 * NSL) * SLAB;
    };
    halfx8 hh8[16], hl8[16];  // the hidden layer, split: 16-unit step k = 2 T + hh of half 0, then of half 1
    static_assert(NSL == 2, "two slices a 128-row weight block: two tiles of the other half activated a slice");

    // wait for slice j (and free slice j - 1's buffer), start slice j + 1's copy; slice j in LDS
    auto next = [&](int j) {
        __builtin_amdgcn_s_waitcnt(0);  // this wavefront's copies of slice j have landed
        __syncthreads();                // everyone's have; slice j - 1's buffer is free
        if (j + 1 < NSLICES) dma_to_lds<THREADS>(slice(j + 1), slab + ((j + 1) & 1) * SLAB, SLAB, tid);
        return static_cast<const uint8_t *>(slab + (j & 1) * SLAB);
    };
    // acc[T] += (rows 32 T .. 32 T + 31 of the slice's weights) B over the slice's CPS 16-column steps
    auto mma = [&](floatx16 (&acc)[4], const uint8_t *sl, const halfx8 *bh, const halfx8 *bl, int rows) {
#pragma unroll
        for (int c = 0; c < CPS; c++)
#pragma unroll
            for (int T = 0; T < 4; T++) {
                const int n = 32 * T + arow;
                const halfx8 ah = *reinterpret_cast<const halfx8 *>(sl + c * 8192 + (g * rows + n) * 16);
                const halfx8 al = *reinterpret_cast<const halfx8 *>(sl + c * 8192 + ((2 + g) * rows + n) * 16);
                acc[T] = mfma16x3(ah, al, bh[c], bl[c], acc[T]);
            }
    };
    // hidden unit of accumulator v of tile T of half h: 128 h + 32 T + 16 (v / 8) + 8 g + v % 8; bias and GELU in
    // place, the running largest magnitude in mx
    const float u1 = ldexpf(1.0f, -(sx + s1));
    auto act = [&](floatx16 &a, int half, int T, float &mx) {
#pragma unroll
        for (int hh = 0; hh < 2; hh++) {
            const float *bp = bias1 + 128 * half + 32 * T + 16 * hh + 8 * g;
            const float4 ba = *reinterpret_cast<const float4 *>(bp), bb = *reinterpret_cast<const float4 *>(bp + 4);
            const float bv[8] = {ba.x, ba.y, ba.z, ba.w, bb.x, bb.y, bb.z, bb.w};
#pragma unroll
            for (int t = 0; t < 8; t++) {
                const float hv = gelu(a[8 * hh + t] * u1 + bv[t]);
                a[8 * hh + t] = hv;
                mx = fmaxf(mx, fabsf(hv));
            }
        }
    };
    // a half of the hidden layer, activated, scaled by its own power of two and split into hh8 / hl8
    auto split_half = [&](floatx16 (&a)[4], float mx, int half) {
        mx = half_max(mx);
        const int sh = shift_for_max(mx);
#pragma unroll
        for (int T = 0; T < 4; T++)
#pragma unroll
            for (int hh = 0; hh < 2; hh++) {
                float hv[8];
#pragma unroll
                for (int t = 0; t < 8; t++) hv[t] = a[T][8 * hh + t];
                split8(hv, ldexpf(1.0f, sh), hh8[8 * half + 2 * T + hh], hl8[8 * half + 2 * T + hh]);
            }
        return sh;
    };

    // The four products run in slice order (W1's two halves, then W2's two halves of hidden units); each one's
    // matrix work overlaps the vector work of the half before it: H^T half 1 = W1 X^T under GELU of half 0, and
    // Y^T = W2 H^T over half 0 under GELU of half 1. Y's sums over the two halves carry the halves' own scales: between
    // them they are rescaled (exactly) to the second's.
    floatx16 acc0[4], acc1[4], y[4];
#pragma unroll
    for (int T = 0; T < 4; T++)
#pragma unroll
        for (int v = 0; v < 16; v++) {
            acc0[T][v] = 0.0f;
            acc1[T][v] = 0.0f;
            y[T][v] = 0.0f;
        }
#pragma unroll
    for (int st = 0; st < NSL; st++) mma(acc0, next(st), xh + CPS * st, xl + CPS * st, 128);
    float m0 = 0.0f;
#pragma unroll
    for (int st = 0; st < NSL; st++) {
        mma(acc1, next(NSL + st), xh + CPS * st, xl + CPS * st, 128);
        act(acc0[2 * st], 0, 2 * st, m0);
        act(acc0[2 * st + 1], 0, 2 * st + 1, m0);
    }
    const int sh0 = split_half(acc0, m0, 0);
    float m1 = 0.0f;
#pragma unroll
    for (int st = 0; st < NSL; st++) {
        mma(y, next(2 * NSL + st), hh8 + CPS * st, hl8 + CPS * st, E);
        act(acc1[2 * st], 1, 2 * st, m1);
        act(acc1[2 * st + 1], 1, 2 * st + 1, m1);
    }
    const int sh1 = split_half(acc1, m1, 1);
    {
        const float r = ldexpf(1.0f, sh1 - sh0);
#pragma unroll
        for (int T = 0; T < 4; T++) y[T] *= r;
    }
#pragma unroll
    for (int st = 0; st < NSL; st++) mma(y, next(3 * NSL + st), hh8 + 8 + CPS * st, hl8 + 8 + CPS * st, E);
    if (!KV && !live) return;
    // output column of accumulator v of tile T: 32 T + 16 (v / 8) + 8 g + v % 8; x += y + b2 (a lane that is not live
    // reads its row's first token, which is there, and stores nothing)
    const float u2 = ldexpf(1.0f, -(sh1 + s2));
#pragma unroll
    for (int T = 0; T < 4; T++)
#pragma unroll
        for (int hh = 0; hh < 2; hh++) {
            const int c0 = 32 * T + 16 * hh + 8 * g;
            float *dst = xrow + c0;
            float rv[8], bv[8], xo[8];
            load8(dst, rv);
            load8(b2 + c0, bv);
#pragma unroll
            for (int t = 0; t < 8; t++) xo[t] = y[T][8 * hh + t] * u2 + bv[t] + rv[t];
            if (live && keep) {
                *reinterpret_cast<float4 *>(dst) = make_float4(xo[0], xo[1], xo[2], xo[3]);
                *reinterpret_cast<float4 *>(dst + 4) = make_float4(xo[4], xo[5], xo[6], xo[7]);
            }
            if constexpr (KV) {
#pragma unroll
                for (int t = 0; t < 8; t++) xv[2 * T + hh][t] = xo[t];
            }
        }
    if constexpr (KV) {
        // the next block's keys (slices 4 NSL ..) then values (6 NSL - NSL ..): 128 outputs each, as four 32-row tiles
        const int sk = norm_split(xv, kn.lnw, kn.lnb, g, xh, xl);
        const float uk = ldexpf(1.0f, -(sk + kn.shift));
#pragma unroll
        for (int part = 0; part < 2; part++) {
            floatx16 a[4];
#pragma unroll
            for (int T = 0; T < 4; T++)
#pragma unroll
                for (int v = 0; v < 16; v++) a[T][v] = 0.0f;
#pragma unroll
            for (int st = 0; st < NSL; st++) mma(a, next(4 * NSL + NSL * part + st), xh + CPS * st, xl + CPS * st, 128);
#pragma unroll
            for (int T = 0; T < 4; T++)
#pragma unroll
                for (int hh = 0; hh < 2; hh++) {
                    const int c0 = 128 * part + 32 * T + 16 * hh + 8 * g;
                    float bv[8], o[8];
                    load8(kn.b + c0, bv);
#pragma unroll
                    for (int t = 0; t < 8; t++) o[t] = a[T][8 * hh + t] * uk + bv[t];
                    if (live) {
                        *reinterpret_cast<float4 *>(kn.out + c0) = make_float4(o[0], o[1], o[2], o[3]);
                        *reinterpret_cast<float4 *>(kn.out + c0 + 4) = make_float4(o[4], o[5], o[6], o[7]);
                    }
                }
        }
    }
}

}  // namespace tah
