// The regression head's reading of a row of predicted quantiles as a distribution (QuantileDist, src/table.rs:
// 292-346), on the card for every row of a member's output at once (src/table.rs:479-486 applies it per row):
// sorted by the total order of f32 (f32::total_cmp), levels i / (n + 1), straight lines between neighbours,
// exponential tails fitted by least squares to the first and last k = clamp(n / 4, 1, 20) points. Per row it
// writes the mean, the sample variance (divisor n - 1), the median (icdf at 0.5) and the icdf at each requested
// level, in f32.
//
// The values are mapped to unsigned keys that order as total_cmp orders the floats (positives with the sign bit set,
// negatives complemented; NaNs after +inf or before -inf by their sign). The sums run in the reference's order --
// left to right over the sorted values, with no contraction of a product into an addition -- so that the moments, the
// median and every quantile between the first and last level come out as the reference computes them; the tails
// take the device logf (within 1 ulp of the host's).
#include <algorithm>

#include "common.hpp"
#include "device_math.hpp"

namespace tah {

constexpr int QS_MAX = 1024;     // values a row at most
constexpr int QS_ALPHAS = 64;    // requested levels at most

// The requested levels, passed to the kernel by value: no copy to the card waits before it.
struct QuantileLevels {
    float v[QS_ALPHAS];
};

__device__ __forceinline__ uint32_t total_order_key(float v) {
    const uint32_t u = __float_as_uint(v);
    return u ^ ((u >> 31) ? 0xFFFFFFFFu : 0x80000000u);
}
__device__ __forceinline__ float from_total_order_key(uint32_t k) {
    return __uint_as_float((k >> 31) ? (k ^ 0x80000000u) : ~k);
}

// f32::clamp: NaN stays NaN (fminf/fmaxf alone would return a bound)
__device__ __forceinline__ float clamp_keep_nan(float x, float lo, float hi) {
    return x != x ? x : fminf(fmaxf(x, lo), hi);
}

// least-squares slope of ys on xs over k points, |.| clamped to [0.01, 100] (src/table.rs:305-310)
__device__ float tail_slope(const float *xs, const float *ys, int k) {
#pragma clang fp contract(off)
    float sx = 0.0f, sy = 0.0f;
    for (int i = 0; i < k; i++) {
        sx += xs[i];
        sy += ys[i];
    }
    const float mx = sx / (float)k, my = sy / (float)k;
    float c = 0.0f, v = 0.0f;
    for (int i = 0; i < k; i++) {
        const float dx = xs[i] - mx;
        c += dx * (ys[i] - my);
        v += dx * dx;
    }
    const float cov = c / (float)k, var = v / (float)k;
    return clamp_keep_nan(fabsf(cov / fmaxf(var, 1e-6f)), 0.01f, 100.0f);
}

__device__ __forceinline__ float level(int i, int n) { return (float)(i + 1) / (float)(n + 1); }

// ---- a wavefront's sort of 64 * K keys held K a lane (position lane * K + r) --------------------------------------
// A bitonic network in its all-ascending form: a merge first compares each position with its mirror in the merged
// block, then at halving strides, so that the lower position always keeps the smaller key.

// The value of lane ^ MASK, through the LDS crossbar, which the sort leaves idle otherwise (with the masks within 16
// lanes as data-parallel moves, a vector instruction a key more: 72 -> 80 us below).
template <int MASK>
__device__ __forceinline__ uint32_t from_lane_xor(uint32_t v) {
    if constexpr (MASK < 32) return __builtin_amdgcn_ds_swizzle(v, (MASK << 10) | 0x1F);
    else return __builtin_amdgcn_ds_bpermute((int)((threadIdx.x & 63) ^ MASK) * 4, v);
}

// The smaller of a and b where bound is 0, the larger where it is all ones.
__device__ __forceinline__ uint32_t keep_side(uint32_t a, uint32_t b, uint32_t bound) {
    uint32_t o;
    asm("v_med3_u32 %0, %1, %2, %3" : "=v"(o) : "v"(a), "v"(b), "v"(bound));
    return o;
}

template <int K>
__device__ __forceinline__ void order(uint32_t (&a)[K], int lo, int hi) {
    const uint32_t x = a[lo], y = a[hi];
    a[lo] = min(x, y);
    a[hi] = max(x, y);
}

// the strides S, S / 2, .. 1 within each lane's keys
template <int K, int S>
__device__ __forceinline__ void lane_strides(uint32_t (&a)[K]) {
    if constexpr (S >= 1) {
#pragma unroll
        for (int r = 0; r < K; r++)
            if (!(r & S)) order(a, r, r + S);
        lane_strides<K, S / 2>(a);
    }
}

// each lane's own K keys in order
template <int K, int SIZE = 2>
__device__ __forceinline__ void lane_sort(uint32_t (&a)[K]) {
    if constexpr (SIZE <= K) {
#pragma unroll
        for (int r = 0; r < K; r++)
            if ((r & (SIZE - 1)) < SIZE / 2) order(a, r, r ^ (SIZE - 1));
        lane_strides<K, SIZE / 4>(a);
        lane_sort<K, SIZE * 2>(a);
    }
}

// the strides of S, S / 2, .. 1 lanes
template <int K, int S>
__device__ __forceinline__ void cross_strides(uint32_t (&a)[K], int lane) {
    if constexpr (S >= 1) {
        const uint32_t bound = (lane & S) ? 0xFFFFFFFFu : 0u;
#pragma unroll
        for (int r = 0; r < K; r++) a[r] = keep_side(a[r], from_lane_xor<S>(a[r]), bound);
        cross_strides<K, S / 2>(a, lane);
    }
}

// merges of G = 2, 4, .. 64 lanes
template <int K, int G = 2>
__device__ __forceinline__ void cross_merge(uint32_t (&a)[K], int lane) {
    if constexpr (G <= 64) {
        const uint32_t bound = (lane & (G / 2)) ? 0xFFFFFFFFu : 0u;
        uint32_t m[K];
#pragma unroll
        for (int r = 0; r < K; r++) m[r] = from_lane_xor<G - 1>(a[K - 1 - r]);
#pragma unroll
        for (int r = 0; r < K; r++) a[r] = keep_side(a[r], m[r], bound);
        cross_strides<K, G / 4>(a, lane);
        lane_strides<K, K / 2>(a);
        cross_merge<K, G * 2>(a, lane);
    }
}

// Up to QS_ROWS rows a workgroup of eight wavefronts; q [rows][n] (n in [2, 64 K]); alphas [na]; stats [rows][3 + na].
//
// Bound by the vector units: a row's sort is about 1,100 instructions of a wavefront (K = 16; a stage between
// registers costs one a key, between lanes the same and an exchange). Each wavefront sorts whole rows in registers, with no barrier, where
// a workgroup sorting one row in LDS waited at each of 55 stages and moved every key through LDS twice in each. The
// sums are one serial chain a row by definition: one wavefront runs all the rows' chains at once, a lane a row, where one
// lane of every row's workgroup had run its own. Meanwhile other wavefronts fit the tails and read the levels, and the
// compute unit's other workgroups sort: with K = 16 eight rows and four workgroups (32 wavefronts) a compute unit; 16
// rows and two workgroups 89 us, 4 rows 77, 32 lanes or 16 a row (fewer exchanges, two or four rows a wavefront)
// 85 and 100. 16,384 rows of 999 and 6 levels: 370 -> 73 us a launch; of 99 10 us.
template <int K, int QS_ROWS, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void k_quantile_stats(int rows, int per, int n, const float *__restrict__ q, int na,
                                                        QuantileLevels alphas, float *__restrict__ stats) {
#pragma clang fp contract(off)
    constexpr int PITCH = 64 * K + 4;  // rows 4 banks apart: 16 rows' 16-byte reads meet no bank twice
    __shared__ __align__(16) float qs[QS_ROWS * PITCH];
    __shared__ float lnx[WAVES - 1][2][20], tails[WAVES - 1][QS_ROWS][4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int row0 = blockIdx.x * per, here = min(per, rows - row0);
    for (int rr = wave; rr < here; rr += WAVES) {
        const float *src = q + (size_t)(row0 + rr) * n;
        uint32_t a[K];
#pragma unroll
        for (int r = 0; r < K; r++) a[r] = r * 64 + lane < n ? total_order_key(src[r * 64 + lane]) : 0xFFFFFFFFu;
        lane_sort<K>(a);
        cross_merge<K>(a, lane);
        float *dst = qs + rr * PITCH + lane * K;
        if constexpr (K >= 4) {
#pragma unroll
            for (int r = 0; r < K; r += 4)
                *reinterpret_cast<float4 *>(dst + r) = make_float4(from_total_order_key(a[r]), from_total_order_key(a[r + 1]),
                                                                   from_total_order_key(a[r + 2]), from_total_order_key(a[r + 3]));
        } else {
#pragma unroll
            for (int r = 0; r < K; r++) dst[r] = from_total_order_key(a[r]);
        }
    }
    __syncthreads();
    const int items = here * (1 + na);
    if (wave == 0) {
        // mean and sample variance, left to right, a lane a row (src/table.rs:322-330); the next eight values are read
        // while these are summed (past n: inside the row's buffer, unused)
        const int row = min(lane, here - 1);
        const float *at = qs + row * PITCH;
        auto sum = [&](auto term) {
#pragma clang fp contract(off)
            float s = 0.0f;
            float4 x = *reinterpret_cast<const float4 *>(at), y = *reinterpret_cast<const float4 *>(at + 4);
            int i = 0;
            for (; i + 8 <= n; i += 8) {
                const float4 x2 = *reinterpret_cast<const float4 *>(at + min(i + 8, 64 * K - 8));
                const float4 y2 = *reinterpret_cast<const float4 *>(at + min(i + 12, 64 * K - 4));
                s += term(x.x); s += term(x.y); s += term(x.z); s += term(x.w);
                s += term(y.x); s += term(y.y); s += term(y.z); s += term(y.w);
                x = x2;
                y = y2;
            }
            for (; i < n; i++) s += term(at[i]);
            return s;
        };
        const float m = sum([](float x) { return x; }) / (float)n;
        const float v = sum([m](float x) {
#pragma clang fp contract(off)
            return (x - m) * (x - m);
        });
        if (lane < here) {
            float *out = stats + (size_t)(row0 + row) * (3 + na);
            out[0] = m;
            out[1] = v / (float)(n - 1);
        }
        return;
    }
    // the levels on as many of the other wavefronts as leave each about 128; each fits the rows' tails for itself
    const int readers = min(WAVES - 1, (items + 127) / 128);
    if (wave > readers) return;
    const int k = max(min(20, n / 4), 1), slot = wave - 1;
    if ((lane & 31) < k) {
        const int i = lane & 31;
        lnx[slot][lane >> 5][i] = logf(fmaxf(lane < 32 ? level(i, n) : 1.0f - level(n - k + i, n), 1e-6f));
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if ((lane >> 1) < here) {
        // a lane a row's tail (src/table.rs:311-315)
        const float *row = qs + (lane >> 1) * PITCH;
        float *t = tails[slot][lane >> 1];
        const int right = lane & 1;
        const float b = tail_slope(lnx[slot][right], right ? row + n - k : row, k);
        if (!right) {
            t[0] = b;
            t[1] = row[0] - b * logf(fmaxf(level(0, n), 1e-6f));
        } else {
            t[2] = -b;
            t[3] = row[n - 1] + b * logf(1.0f - fminf(level(n - 1, n), 1.0f - 1e-6f));
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    // icdf at 0.5 and at each of alphas, an item a lane (src/table.rs:333-345)
    for (int item = slot * 64 + lane; item < items; item += readers * 64) {
        const int rr = item / (1 + na), which = item - rr * (1 + na);
        const float *row = qs + rr * PITCH, *t = tails[slot][rr];
        const float alpha = which == 0 ? 0.5f : alphas.v[which - 1];
        float y;
        if (alpha < level(0, n)) {
            y = t[0] * logf(fmaxf(alpha, 1e-6f)) + t[1];
        } else if (alpha > level(n - 1, n)) {
            y = t[2] * logf(fmaxf(1.0f - alpha, 1e-6f)) + t[3];
        } else if (alpha >= level(n - 1, n)) {
            y = row[n - 1];
        } else {
            // the number of levels[0 .. n - 2] at most alpha, less one (the segment's left end), within [0, n - 2]
            int lo = 0, hi = n - 1;
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (level(mid, n) <= alpha) lo = mid + 1;
                else hi = mid;
            }
            const int i = min(max(lo - 1, 0), n - 2);
            const float f = clamp_keep_nan((alpha - level(i, n)) / fmaxf(level(i + 1, n) - level(i, n), 1e-6f), 0.0f, 1.0f);
            y = row[i] + f * (row[i + 1] - row[i]);
        }
        stats[(size_t)(row0 + rr) * (3 + na) + 2 + which] = y;
    }
}

template <int K>
static void launch_quantile_stats(hipStream_t s, int rows, int n, const float *q, int na, const QuantileLevels &alphas,
                                  float *stats) {
    // as many rows a workgroup as leave four workgroups' LDS on a compute unit (at most the tails' 32), once there are
    // rows for two workgroups a compute unit of one row each
    constexpr int ROWS = K == 16 ? 8 : K == 8 ? 16 : 32;
    const int per = std::min(ROWS, rows / 512 + (rows % 512 > 0));
    // at most 2^31 threads a launch (33 million rows of eight a workgroup)
    const int most = per << 22;
    for (int r0 = 0; r0 < rows;) {
        const int here = std::min(most, rows - r0);
        hipLaunchKernelGGL((k_quantile_stats<K, ROWS, 8>), dim3(here / per + (here % per > 0)), dim3(512), 0, s, here, per, n,
                           q + (size_t)r0 * n, na, alphas, stats + (size_t)r0 * (3 + na));
        r0 += here;
    }
    TAH_LAUNCHED();
}

// alphas [na] in host memory.
void quantile_stats(hipStream_t s, int rows, int n, const float *q, int na, const float *alphas, float *stats) {
    if (rows <= 0) return;
    if (n < 2 || n > QS_MAX || na < 0 || na > QS_ALPHAS || (na > 0 && !alphas))
        throw ArgError{"quantile_stats: 2 to 1024 quantiles a row and at most 64 levels"};
    QuantileLevels lv{};
    std::copy(alphas, alphas + na, lv.v);
    // the fewest keys a lane that hold a row: a sort's work grows with them, the padding past n included
    if (n <= 128) launch_quantile_stats<2>(s, rows, n, q, na, lv, stats);
    else if (n <= 256) launch_quantile_stats<4>(s, rows, n, q, na, lv, stats);
    else if (n <= 512) launch_quantile_stats<8>(s, rows, n, q, na, lv, stats);
    else launch_quantile_stats<16>(s, rows, n, q, na, lv, stats);
}

}  // namespace tah
