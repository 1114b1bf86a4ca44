// The row stage's fused block: a table row's tokens through attention, output projection and feed-forward in one kernel.
// A kernel for every count of key tiles: row_block.hip launches them, row_block_next4.hip and row_block_next8.hip hold
// those that form the next block's keys and values (a source each, since each kernel takes seconds to compile).
#pragma once

#include <algorithm>

#include "attend.hpp"
#include "ff128.hpp"

namespace tah {

// ---- fused row block, attention half ------------------------------------------------------------------------------
// x += out(attend(rope(Wq layer_norm1(x) + bq) / 4, rope(K), V)) + bo for every token of one row over all the row's
// tokens (src/nn.rs:357-419, Rope src/nn.rs:304-321), for e = 128, 8 heads of 16 and T <= 32 W tokens; the keys and
// values [T][2 e] (k then v per token, without rotation) come from a projection before it.
// grid ceil(n / R); W = 4 or 8 wavefronts for R rows (two of up to 64 tokens, else one), NTL key tiles of 32 a row:
// wavefront w owns tokens 32 (w % (W / R)) + 0..31 of row w / (W / R) of the workgroup's, lane l token l % 32, as the B
// operand of every product (as in k_cell_block):
//  * the query projection as in k_cell_block, its accumulators rotated in registers (a coordinate's partner for the
//    rotation sits on lane l ^ 32) and scaled by 1 / sqrt(16), then split, each head's at its own power of two;
//  * per head the workgroup stages its rows' keys (rotated) and values into LDS split into fp16 halves, scaled by the
//    head's power of two (a maximum over the row's tokens, across wavefronts through LDS): half the threads a key
//    each, the others two coordinates of eight values. Staging runs two heads ahead, its loads three: their maxima are
//    formed behind a head's attention, under which they land (formed where the loads were issued, each head waited for
//    memory: 60% of the wavefronts' cycles);
//  * slots past a row's tokens hold its last key again, zero values and zero ones, so that no score is masked;
//  * the attention of attend.hpp, above four tiles in two groups, and the output projection run as in k_cell_block.
// With FF the block's feed-forward half follows in the same kernel, as in k_cell_block; with KV as well the next
// row block's keys and values (kn.out [n][T][2 e], which may be kv itself: a workgroup reads only its own row's keys
// and values, all of them before its feed-forward half starts).
//
// W = 8 takes rows of 129 to 256 tokens, one workgroup a compute unit (two wavefronts a SIMD, as two workgroups of W =
// 4). Measured with KV: 500 rows of 204 tokens 265 us a launch with the eight wavefronts (480 with the projection, the
// rotation, the f32-MFMA attention, the output projection and the feed-forward apart). R = 2: 389 rows of 41 tokens 84
// us as 389 workgroups, 64 us as 195.
template <bool FF, bool KV, int W, int R, int NTL>
__global__ __launch_bounds__(64 * W, 2) void k_row_block(int n, int T, int keep, float *tok, const float *kv,
                                                       const float *__restrict__ cosv, const float *__restrict__ sinv,
                                                       const float *__restrict__ n1w, const float *__restrict__ n1b,
                                                       const uint8_t *__restrict__ qimg, int qshift,
                                                       const float *__restrict__ qb, const uint8_t *__restrict__ oimg,
                                                       int oshift, const float *__restrict__ ob, const float *__restrict__ n2w, const float *__restrict__ n2b,
                                                       const uint8_t *__restrict__ w1img, const float *__restrict__ b1,
                                                       int s1, const uint8_t *__restrict__ w2img,
                                                       const float *__restrict__ b2, int s2, KvNext kn) {
    static_assert(FF || !KV, "the next block's keys and values come from the feed-forward's registers");
    static_assert((W == 4 && (R == 1 || R == 2)) || (W == 8 && R == 1), "a half wave group a row at least");
    constexpr int E = 128, THREADS = 64 * W, NT = 32 * W;  // NT: token slots
    constexpr int PER = NT / R, RW = W / 2 / R;            // slots a row, staging wavefronts a row (of each half)
    constexpr int STAGED = NT * 128;                       // a staged head: keys and values, hi and lo
    constexpr int PAD = 3 * STAGED;                        // behind the three staged heads (after the query weights)
    static_assert(NTL >= 1 && 32 * NTL <= PER, "a row's key tiles");
    __shared__ __align__(1024) uint8_t lds[65536 < PAD + 2 * NT * 32 ? PAD + 2 * NT * 32 : 65536];
    __shared__ __align__(16) float ffb[FF ? 256 : 4];  // FF: the first feed-forward layer's bias
    __shared__ __align__(16) float qbs[128];
    __shared__ __align__(16) float cst[2][PER][8];  // cos, sin of token t, pair k
    __shared__ float red[3][2][W / 2];              // [head % 3][keys, values][wavefront of the half]
    __shared__ int shs[3][2][R];                    // [buffer][keys, values][row]: the staged head's scales
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r32 = lane & 31, g = lane >> 5;
    const int rs = wave / (W / R);  // this wavefront's row of the workgroup's
    const int row = min((int)blockIdx.x * R + rs, n - 1);
    const int tk = (wave % (W / R)) * 32 + r32;  // this lane's token
    const bool live = tk < T && (int)blockIdx.x * R + rs < n;
    float *xrow = tok + ((size_t)row * T + (live ? tk : 0)) * E;
    dma_to_lds<THREADS>(qimg, lds, 65536, tid);
    if (tid < 32) reinterpret_cast<float4 *>(qbs)[tid] = *reinterpret_cast<const float4 *>(qb + 4 * tid);
    if (tid < T) {
#pragma unroll
        for (int k = 0; k < 8; k++) {
            cst[0][tid][k] = cosv[tid * 8 + k];
            cst[1][tid][k] = sinv[tid * 8 + k];
        }
    }

    // staging of head h: thread t < NT takes slot t's key (16 coordinates, rotated; slots past the row's tokens its last
    // key again, so that scores need no mask: their values and ones are zero), thread NT + t coordinates 2 (t % 8) and
    // the next of the eight slots 8 (t / 8) ..: whole 16-byte entries of V^T
    const bool st_key = tid < NT;
    const int st_slot = st_key ? tid : (tid - NT) & ~7, st_row = st_slot / PER, st_tok = st_slot % PER;
    const int st_c = 2 * (tid & 7);
    // eight pairs of floats a thread, from addresses that are always the row's (no load sits behind a branch, where each
    // would be waited for by itself): a key's in order, or a pair of each value's, past the last token its again
    const float *st_src = kv + ((size_t)min((int)blockIdx.x * R + st_row, n - 1) * T + min(st_tok, T - 1)) * 2 * E +
                          (st_key ? 0 : E + st_c);
    const int st_step = st_key ? 2 : 2 * E, st_last = st_key ? 7 : max(T - 1 - st_tok, 0);
    auto stage_load = [&](int h, float (&stv)[16]) {
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float2 a = *reinterpret_cast<const float2 *>(st_src + 16 * h + min(i, st_last) * st_step);
            stv[2 * i] = a.x;
            stv[2 * i + 1] = a.y;
        }
    };
    auto stage_max = [&](const float (&stv)[16], int par) {
        float mx = 0.0f;
#pragma unroll
        for (int c = 0; c < 16; c++) mx = fmaxf(mx, fabsf(stv[c]));
        mx = wave_max(mx);
        if (lane == 0) red[par][wave / (W / 2)][wave & (W / 2 - 1)] = mx;
    };
    auto stage_store = [&](const float (&stv)[16], int par, int buf) {
        // the keys' maximum is over the unrotated values: rotation keeps each pair's norm, so the rotated values stay
        // within sqrt(2) of it, and the split's scale (a maximum below 2^14) leaves that room
        const int part = st_key ? 0 : 1;
        float mx = red[par][part][st_row * RW];
#pragma unroll
        for (int i = 1; i < RW; i++) mx = fmaxf(mx, red[par][part][st_row * RW + i]);
        const int s = shift_for_max(mx * 1.5f);
        const float f = ldexpf(1.0f, s);
        if (st_tok == 0) shs[buf][part][st_row] = s;
        uint8_t *const at = lds + buf * STAGED;
        if (st_key) {
            float c[8], sn[8], rk[16];
            load8(cst[0][min(st_tok, T - 1)], c);
            load8(cst[1][min(st_tok, T - 1)], sn);
#pragma unroll
            for (int k = 0; k < 8; k++) {
                rk[k] = stv[k] * c[k] - stv[k + 8] * sn[k];
                rk[k + 8] = stv[k + 8] * c[k] + stv[k] * sn[k];
            }
#pragma unroll
            for (int i = 0; i < 2; i++) {
                halfx8 hi, lo;
                split8(rk + 8 * i, f, hi, lo);
                *reinterpret_cast<halfx8 *>(at + (i * NT + st_slot) * 16) = hi;
                *reinterpret_cast<halfx8 *>(at + NT * 32 + (i * NT + st_slot) * 16) = lo;
            }
        } else {
            const int tg = st_slot >> 3;
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const int cd = st_c + i, rw = ((cd & 3) | ((cd & 4) << 1) | ((cd & 8) >> 1)) ^ (tg & 15);
                float v[8];
#pragma unroll
                for (int t = 0; t < 8; t++) v[t] = st_tok + t < T ? stv[2 * t + i] : 0.0f;
                halfx8 hi, lo;
                split8(v, f, hi, lo);
                *reinterpret_cast<halfx8 *>(at + NT * 64 + (tg * 16 + rw) * 16) = hi;
                *reinterpret_cast<halfx8 *>(at + NT * 96 + (tg * 16 + rw) * 16) = lo;
            }
        }
    };
    float st0[16], st1[16], st2[16];  // heads 0 to 2
    stage_load(0, st0);
    stage_load(1, st1);
    stage_load(2, st2);
    __builtin_amdgcn_sched_barrier(0);

    // this wavefront's tokens: layer norm, then split as the B operand (coordinates 16 ks + 8 g + t)
    float xv[8][8];
#pragma unroll
    for (int ks = 0; ks < 8; ks++) load8(xrow + 16 * ks + 8 * g, xv[ks]);  // past the tokens the first's, used for nothing
    {
        float sum = 0.0f;
#pragma unroll
        for (int ks = 0; ks < 8; ks++)
#pragma unroll
            for (int t = 0; t < 8; t++) sum += xv[ks][t];
        sum = half_sum(sum);
        const float mean = sum / 128.0f;
        float sq = 0.0f;
#pragma unroll
        for (int ks = 0; ks < 8; ks++)
#pragma unroll
            for (int t = 0; t < 8; t++) {
                const float dv = xv[ks][t] - mean;
                sq += dv * dv;
            }
        sq = half_sum(sq);
        const float inv = 1.0f / sqrtf(sq / 128.0f + 1e-5f);
#pragma unroll
        for (int ks = 0; ks < 8; ks++) {
            float wv[8], bv[8];
            load8(n1w + 16 * ks + 8 * g, wv);
            load8(n1b + 16 * ks + 8 * g, bv);
#pragma unroll
            for (int t = 0; t < 8; t++) xv[ks][t] = (xv[ks][t] - mean) * inv * wv[t] + bv[t];
        }
    }
    float xmax = 0.0f;
#pragma unroll
    for (int ks = 0; ks < 8; ks++)
#pragma unroll
        for (int t = 0; t < 8; t++) xmax = fmaxf(xmax, fabsf(xv[ks][t]));
    xmax = half_max(xmax);
    const int sx = shift_for_max(xmax);

    // query projection (accumulator v of tile T: head 2 T + v / 8, coordinate 8 g + v % 8), bias, rotation, 1 / 4
    floatx16 qa[4];
    {
        const int arow = sigma32(r32);
        halfx8 xh[8], xl[8];
#pragma unroll
        for (int ks = 0; ks < 8; ks++) split8(xv[ks], ldexpf(1.0f, sx), xh[ks], xl[ks]);
#pragma unroll
        for (int T4 = 0; T4 < 4; T4++)
#pragma unroll
            for (int v = 0; v < 16; v++) qa[T4][v] = 0.0f;
        stage_max(st0, 0);
        stage_max(st1, 1);
        stage_max(st2, 2);
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();  // the query weights, bias and rotation tables are in LDS; the first heads' maxima in red
#pragma unroll
        for (int ks = 0; ks < 8; ks++)
#pragma unroll
            for (int T4 = 0; T4 < 4; T4++) {
                const int nn = 32 * T4 + arow;
                const halfx8 ah = *reinterpret_cast<const halfx8 *>(lds + ks * 8192 + (g * 128 + nn) * 16);
                const halfx8 al = *reinterpret_cast<const halfx8 *>(lds + ks * 8192 + ((2 + g) * 128 + nn) * 16);
                qa[T4] = mfma16x3(ah, al, xh[ks], xl[ks], qa[T4]);
            }
        __builtin_amdgcn_sched_barrier(0);
        const float u = ldexpf(1.0f, -(sx + qshift));
        const int ct = live ? tk : 0;
        float cs[8], sn[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            cs[k] = cst[0][ct][k];
            sn[k] = cst[1][ct][k];
        }
        const float sgn = g == 0 ? -1.0f : 1.0f;
#pragma unroll
        for (int T4 = 0; T4 < 4; T4++)
#pragma unroll
            for (int hh = 0; hh < 2; hh++) {
                float bv[8];
                load8(qbs + 32 * T4 + 16 * hh + 8 * g, bv);
#pragma unroll
                for (int t = 0; t < 8; t++) {
                    const float qv = qa[T4][8 * hh + t] * u + bv[t];
                    const auto sw2 = __builtin_amdgcn_permlane32_swap(__float_as_uint(qv), __float_as_uint(qv), false, false);
                    const float other = __uint_as_float(g ? sw2[0] : sw2[1]);  // the coordinate 8 away, lane l ^ 32
                    qa[T4][8 * hh + t] = (qv * cs[t] + sgn * other * sn[t]) * 0.25f;
                }
            }
    }
    // the queries, each head's split at its own power of two, as in k_cell_block
    halfx8 qh[8], ql[8];
    HeadShifts sq;
#pragma unroll
    for (int h = 0; h < 8; h++) {
        float qv[8], qmax = 0.0f;
#pragma unroll
        for (int t = 0; t < 8; t++) {
            qv[t] = qa[h >> 1][8 * (h & 1) + t];
            qmax = fmaxf(qmax, fabsf(qv[t]));
        }
        const int s = min(shift_for_max(half_max(qmax)), 127);
        sq.set(h, s);
        split8(qv, ldexpf(1.0f, s), qh[h], ql[h]);
    }
    sq.pack();
    __syncthreads();  // everyone is done with the query weights
    pad_rows<NT>(lds + PAD, tid, PER, T);
    stage_store(st0, 0, 0);
    stage_store(st1, 1, 1);
    stage_store(st2, 2, 2);
    float stv[16];
    const int arow = sigma32(r32);
    const bool one = (r32 & 27) == 16;  // as in k_cell_block; a row's V^T steps start at PER / 16 times its number
    const int vstep = one ? 0 : STAGED, kb = (g * NT + rs * PER + arow) * 16;
    const int vb = (one ? PAD + 16 * g : NT * 64 + 256 * g + 16 * ((r32 & 15) ^ g ^ (R == 2 ? 8 * rs : 0))) +
                   rs * (PER * 32 + (one ? 128 : 0));
    constexpr int NA = NTL < 4 ? NTL : 4, NB = NTL - NA;  // a head's key tiles, as one group of up to four or two
    floatx16 sc[NA];
    // the heads' outputs, split as the output projection's input at the least of the value scales of the heads up to theirs
    halfx8 oh[8], ol[8];
    int so[8];
#pragma unroll
    for (int h = 0; h < 8; h++) {
        const int buf = h % 3, nbuf = (h + 1) % 3;
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();  // head h + 1 is staged, head h + 2's maxima are in red; everyone is done with head h - 1
        if (h == 0) {
#pragma unroll
            for (int j = 0; j < NA; j++) sc[j] = score_tile<NT>(lds + kb, j, qh[0], ql[0]);
        }
        // two heads ahead: head h + 2 into the buffer head h - 1 used, then head h + 3's values into registers (their
        // maxima are formed behind this head's attention, under which the loads land)
        if (h >= 1 && h + 2 < 8) stage_store(stv, (h + 2) % 3, (h + 2) % 3);
        if (h + 3 < 8) {
            stage_load(h + 3, stv);
            __builtin_amdgcn_sched_barrier(0);  // the loads go out here
        }
        // behind the last staged head the output projection's weights, 16-column steps of 8 KB in the heads' order: W = 8,
        // 0..3 and 4..7 into the buffers of heads 5 and 6; W = 4, 0 past the ones, 1, 2 and 3, 4 into those buffers
        if constexpr (W == 8) {
            if (h >= 6) dma_to_lds<THREADS>(oimg + (h - 6) * 32768, lds + (h == 6 ? 2 : 0) * STAGED, 32768, tid);
        } else {
            if (h == 5) dma_to_lds<THREADS>(oimg, lds + 57344, 8192, tid);
            if (h == 6) dma_to_lds<THREADS>(oimg + 8192, lds + 32768, 16384, tid);
            if (h == 7) dma_to_lds<THREADS>(oimg + 24576, lds, 16384, tid);
        }
        const float to_log2 = ldexpf(LOG2E, -(shs[buf][0][rs] + sq.get(h)));
        const int svh = __builtin_amdgcn_readfirstlane(shs[buf][1][rs]);  // a wavefront's tokens are one row's
        so[h] = h ? min(so[h - 1], svh) : svh;
        float ref;
        floatx16 o;
        const uint8_t *kn0 = lds + nbuf * STAGED + kb;
        auto ahead = [&](int j) {
            if (h + 1 < 8) sc[j] = score_tile<NT>(kn0, j, qh[(h + 1) & 7], ql[(h + 1) & 7]);
        };
        const int vbh = vb + buf * vstep;
        if constexpr (NB == 0) {
            attend_tiles<NT, NA, true>(sc, to_log2, lds, vbh, ref, o, ahead);
        } else {
            const uint8_t *kb1 = lds + buf * STAGED + kb;
            attend_tiles<NT, NA, true>(sc, to_log2, lds, vbh, ref, o, [&](int j) {
                if (j < NB) sc[j] = score_tile<NT>(kb1, NA + j, qh[h], ql[h]);
            });
            attend_tiles<NT, NB, false>(sc, to_log2, lds, vbh + NA * 1024, ref, o, ahead);
#pragma unroll
            for (int j = NB; j < NA; j++) ahead(j);
        }
        const float f = ldexpf(1.0f, so[h] - svh) / o[8];
        float ov[8];
#pragma unroll
        for (int t = 0; t < 8; t++) ov[t] = o[t] * f;
        split8(ov, 1.0f, oh[h], ol[h]);
        if (h + 3 < 8) stage_max(stv, (h + 3) % 3);
    }
    // output projection
    floatx16 acc[4];
    {
#pragma unroll
        for (int T4 = 0; T4 < 4; T4++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[T4][v] = 0.0f;
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();  // everyone is done with the staged heads; the weights copied through the last heads have landed
        if (W == 4) {
            dma_to_lds<THREADS>(oimg + 40960, lds + 16384, 16384, tid);
            dma_to_lds<THREADS>(oimg + 57344, lds + 49152, 8192, tid);
        }
        constexpr int AT[8] = {57344, 32768, 40960, 0, 8192, 16384, 24576, 49152};  // W = 4: where each step is
#pragma unroll
        for (int ks = 0; ks < 8; ks++) {
            if (W == 4 && ks == 5) {
                __builtin_amdgcn_s_waitcnt(0);
                __syncthreads();  // the rest of the weights
            }
            if (ks > 0) lower_scale(acc, so[ks - 1], so[ks]);
            const uint8_t *ws = lds + (W == 4 ? AT[ks] : ks < 4 ? 2 * STAGED + ks * 8192 : (ks - 4) * 8192);
#pragma unroll
            for (int T4 = 0; T4 < 4; T4++) {
                const int nn = 32 * T4 + arow;
                const halfx8 ah = *reinterpret_cast<const halfx8 *>(ws + (g * 128 + nn) * 16);
                const halfx8 al = *reinterpret_cast<const halfx8 *>(ws + ((2 + g) * 128 + nn) * 16);
                acc[T4] = mfma16x3(ah, al, oh[ks], ol[ks], acc[T4]);
            }
        }
    }
    if (!FF && !live) return;
    const float u = ldexpf(1.0f, -(so[7] + oshift));
    float xn[8][8];  // the new values as the feed-forward's input: columns 16 ks + 8 g + t
#pragma unroll
    for (int T4 = 0; T4 < 4; T4++)
#pragma unroll
        for (int hh = 0; hh < 2; hh++) {
            const int n0 = 32 * T4 + 16 * hh + 8 * g;
            float bv[8], xr[8];
            load8(ob + n0, bv);
            load8(xrow + n0, xr);
#pragma unroll
            for (int t = 0; t < 8; t++) xn[2 * T4 + hh][t] = xr[t] + acc[T4][8 * hh + t] * u + bv[t];
            if (live) {
                *reinterpret_cast<float4 *>(xrow + n0) = make_float4(xn[2 * T4 + hh][0], xn[2 * T4 + hh][1],
                                                                     xn[2 * T4 + hh][2], xn[2 * T4 + hh][3]);
                *reinterpret_cast<float4 *>(xrow + n0 + 4) = make_float4(xn[2 * T4 + hh][4], xn[2 * T4 + hh][5],
                                                                         xn[2 * T4 + hh][6], xn[2 * T4 + hh][7]);
            }
        }
    if constexpr (FF) {
        __syncthreads();  // every wavefront is done with the attention's LDS (no copy is in flight after head 7)
        ff128_start<THREADS>(lds, ffb, w1img, b1, tid);
        if constexpr (KV) {
            kn.out += ((size_t)row * T + (live ? tk : 0)) * 2 * E;
            ff128_rows<true, THREADS>(xn, live, xrow, lds, ffb, n2w, n2b, w1img, s1, w2img, b2, s2, tid, kn, tk < keep);
        } else {
            ff128_rows<false, THREADS>(xn, live, xrow, lds, ffb, n2w, n2b, w1img, s1, w2img, b2, s2, tid);
        }
    }
}

// What a launch takes besides its shape.
struct RowLaunch {
    hipStream_t s;
    int n, T, keep;
    float *tok;
    const float *kv, *cosv, *sinv;
    const DevBlock &b;
    KvNext kn;
};

// With the feed-forward half and the next block's keys and values.
template <int W, int R, int NTL>
void launch_row_next(const RowLaunch &a) {
    const DevBlock &b = a.b;
    hipLaunchKernelGGL((k_row_block<true, true, W, R, NTL>), dim3((a.n + R - 1) / R), dim3(64 * W), 0, a.s, a.n, a.T, a.keep,
                       a.tok, a.kv, a.cosv, a.sinv, b.n1w, b.n1b, b.inimg, b.ins, b.in_b, b.outimg, b.outs, b.out_b, b.n2w,
                       b.n2b, b.l1img, b.l1b, b.l1s, b.l2img, b.l2b, b.l2s, a.kn);
}

}  // namespace tah
