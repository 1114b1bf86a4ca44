// Attention of 32 columns a wavefront over keys staged in LDS, on the fp16 matrix cores with split f32 operands: the part
// that the fused column and row blocks and the inducing points' attention of a fit share.
#pragma once

#include "device_math.hpp"

namespace tah {

// A head's keys and values are staged in LDS as fp16 halves for NT key slots (16 dims): keys [dims half][slot][8] hi
// then lo, V^T [16-slot step][8-slot half][row][8] hi then lo (NT x 32 bytes each, NT x 128 in all). S^T = K Q^T and
// O^T = V^T P^T, the lane's column (cell or token) l % 32.
//
// Bound by vector instructions (an exp2, its argument and two splits a score, 4 cycles each and 16 for the exp2) with
// the matrix work beside them, so the order is what counts: a head is one straight run of instructions (no running
// maximum and its branches: all NTL tiles' scores are formed first), the next head's scores are formed a tile at a time
// between this head's weights, and each 16-key step's two value operands are read a step ahead, so that no product
// waits for LDS. The outputs go where the head's queries were, and the output projection runs once behind all heads
// (its sums would hold 64 registers through them).
//
// V^T has 16 rows and the product takes 32: lanes r32 = 16 and 20 read rows of ones for the row's own keys (PAD, one
// 16-byte entry a step and 8-slot half, where the step's swizzle finds it, its lo rows zero), whose sums in accumulator
// 8 are the weights' sum; the other lanes past 15 read any row (their sums are not used).
// pad: 2 NT x 32 bytes; keys of a row take the slots [i per, i per + T) (i: the row), the other slots' ones are zero.
template <int NT>
__device__ __forceinline__ void pad_rows(uint8_t *pad, int tid, int per, int T) {
    if (tid < NT / 8) {  // 8-slot group: step tid / 2, half tid % 2
        const int st = tid >> 1, at = 512 * st + 32 * (st & 7) + 16 * (tid & 1);
        uint32_t w[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int k = (8 * tid + 2 * i) % per;
            w[i] = (k < T ? 0x3c00u : 0u) | (k + 1 < T ? 0x3c000000u : 0u);
        }
        *reinterpret_cast<uint4 *>(pad + at) = make_uint4(w[0], w[1], w[2], w[3]);
        *reinterpret_cast<uint4 *>(pad + NT * 32 + at) = make_uint4(0u, 0u, 0u, 0u);
    }
}

// The shifts of eight heads' queries, four to a register (held through all heads, where a register a head meant spills).
// From -128 to 127 (14 - 128 is the least there is).
struct HeadShifts {
    int w[2] = {0, 0};
    __device__ __forceinline__ void set(int h, int shift) { w[h >> 2] |= (shift & 255) << (8 * (h & 3)); }
    // behind the last set: the compiler would otherwise keep the eight shifts it packed
    __device__ __forceinline__ void pack() { asm volatile("" : "+v"(w[0]), "+v"(w[1])); }
    __device__ __forceinline__ int get(int h) const { return (int)(int8_t)(w[h >> 2] >> (8 * (h & 3))); }
};

// The output projection's sums from the input scale 2^from to 2^to (the same in every lane, to <= from).
__device__ __forceinline__ void lower_scale(floatx16 (&acc)[4], int from, int to) {
    if (to == from) return;
    const float r = ldexpf(1.0f, to - from);
#pragma unroll
    for (int T = 0; T < 4; T++) acc[T] *= r;
}

template <int NT>
__device__ __forceinline__ floatx16 score_tile(const uint8_t *kb, int j, halfx8 qh, halfx8 ql) {
    const halfx8 ah = *reinterpret_cast<const halfx8 *>(kb + 512 * j);
    const halfx8 al = *reinterpret_cast<const halfx8 *>(kb + 512 * j + NT * 32);
    floatx16 z;
#pragma unroll
    for (int v = 0; v < 16; v++) z[v] = 0.0f;
    return mfma16x3(ah, al, qh, ql, z);
}

// TILES tiles of 32 keys of a head from their scores sc (log2 units once times to_log2) into o: O^T (accumulators
// 0..7: the lane's coordinates 8 g + 0..7 times the values' scale, 8: the weights' sum), the weights 2^(score - ref +
// 12). FIRST sets ref and o, the tiles after raise them. vb: this lane's offset in lds of the tiles' V^T hi rows before
// the step's swizzle (bits 5..7). next(j) runs behind tile j: it may form another tile's scores in sc[j].
template <int NT, int TILES, bool FIRST, int S, class F>
__device__ __forceinline__ void attend_tiles(floatx16 (&sc)[S], float to_log2, const uint8_t *lds, int vb, float &ref,
                                             floatx16 &o, F &&next) {
    static_assert(TILES <= S && TILES <= 4, "the swizzle's period is eight steps");
    auto vload = [&](int st, halfx8 &vh, halfx8 &vl) {
        const uint8_t *a = lds + (vb ^ (32 * st)) + 512 * st;
        vh = *reinterpret_cast<const halfx8 *>(a);
        vl = *reinterpret_cast<const halfx8 *>(a + NT * 32);
    };
    halfx8 vh, vl;
    vload(0, vh, vl);
    float mx = sc[0][0];
#pragma unroll
    for (int j = 0; j < TILES; j++)
#pragma unroll
        for (int v = 0; v < 16; v++) mx = fmaxf(mx, sc[j][v]);
    mx = half_max(mx) * to_log2;
    if (FIRST) {
        ref = mx;
#pragma unroll
        for (int v = 0; v < 16; v++) o[v] = 0.0f;
    } else {
        mx = fmaxf(mx, ref);
        o *= exp2_hw(ref - mx);
        ref = mx;
    }
    const float off = 12.0f - ref;
#pragma unroll
    for (int st = 0; st < 2 * TILES; st++) {
        halfx8 nh = vh, nl = vl;
        if (st + 1 < 2 * TILES) vload(st + 1, nh, nl);
        float p[8];
#pragma unroll
        for (int t = 0; t < 8; t++) p[t] = exp2_hw(fmaf(sc[st >> 1][8 * (st & 1) + t], to_log2, off));
        halfx8 ph, pl;
        split8(p, 1.0f, ph, pl);
        o = mfma16x3(vh, vl, ph, pl, o);
        vh = nh;
        vl = nl;
        if (st & 1) next(st >> 1);
    }
}

}  // namespace tah
