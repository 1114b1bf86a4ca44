// The column and row stages of a fit on the card (the reference's Attend::columns and Attend::rows,
// src/fit.rs:54-65, with the CPU loops they replace at src/fit.rs:326-423 and src/fit.rs:486-540), keeping the
// cells resident between the two stages.
//
// Per batch of feature groups (cells [groups][rows][e], group-major so each group's cells are contiguous):
// input layer and target embedding (per label digit), then per column block: the inducing points' queries attend
// to the group's cells (k_ind_attn16: online softmax over blocks of 128 cells, split-fp16 MFMA, split over key ranges
// and merged as in the in-context attention), the inducing points' output projection and feed-forward, their keys
// and values for the second attention written straight into the column cache layout, and the cells' own block
// against them (column_block, shared with prediction).
#include <algorithm>

#include "attend.hpp"
#include "common.hpp"

namespace tah {

static dim3 blocks_of(size_t count) { return dim3((unsigned)((count + 255) / 256)); }

// cells [gb][rows][e] of feature groups g0.. through the input layer, with y (one label digit) its target's embedding
// added as k_add_y adds it. Bound by the cells' way to memory: four coordinates a thread for FIT_ROWS rows of group
// blockIdx.y, G = group's weights in registers (G = 0: any group size, read again for each row). 1,000,000 cells: 680 us
// with a float a thread and 400 for the embedding's pass, 592 with four floats and
// their weights read for every cell, 170 so.
constexpr int FIT_ROWS = 64;
template <int G>
__global__ __launch_bounds__(256) void k_fit_cells(int rows, int features, int g0, int group, int e,
                                                    const float *__restrict__ x, const float *__restrict__ in_w,
                                                    const float *__restrict__ in_b, const float *__restrict__ y,
                                                    int max_classes, const float *__restrict__ table,
                                                    float *__restrict__ cells) {
    const int n = G ? G : group, e4 = e / 4, wide = min(e4, 256), side = 256 / wide;  // rows side by side
    const int rl = (int)threadIdx.x / wide, g = g0 + (int)blockIdx.y;
    if (rl >= side) return;
    const int r1 = min(rows, ((int)blockIdx.x + 1) * FIT_ROWS);
    int from[8];
#pragma unroll
    for (int k = 0; k < (G ? G : 8); k++) from[k] = k < n ? (g + (1 << k)) % features : 0;
    for (int o = 4 * ((int)threadIdx.x - rl * wide); o < e; o += 4 * wide) {
        float w[4][G ? G : 1], b[4];
#pragma unroll
        for (int c = 0; c < 4; c++) {
            b[c] = in_b[o + c];
#pragma unroll
            for (int k = 0; k < G; k++) w[c][k] = in_w[(o + c) * G + k];
        }
        for (int r = blockIdx.x * FIT_ROWS + rl; r < r1; r += side) {
            const float *xr = x + (size_t)r * features;
            float vals[8];
            bool missing = true;
#pragma unroll
            for (int k = 0; k < (G ? G : 8); k++)
                if (k < n) {
                    vals[k] = xr[from[k]];
                    missing = missing && vals[k] == -100.0f;
                }
            float out[4];
#pragma unroll
            for (int c = 0; c < 4; c++) {
                float s = 0.0f;
#pragma unroll
                for (int k = 0; k < (G ? G : 8); k++)
                    if (k < n) s += (G ? w[c][G ? k : 0] : in_w[(o + c) * group + k]) * vals[k];
                out[c] = missing ? -100.0f : s + b[c];
            }
            if (y) {
                const float yr = y[r];
                const float *t = max_classes > 0 ? table + (size_t)(int)yr * e : table;
#pragma unroll
                for (int c = 0; c < 4; c++) out[c] += max_classes > 0 ? t[o + c] : t[o + c] * yr + t[e + o + c];
            }
            *reinterpret_cast<float4 *>(cells + ((size_t)blockIdx.y * rows + r) * e + o) =
                make_float4(out[0], out[1], out[2], out[3]);
        }
    }
}

// cells [gb][rows][e] += the target's embedding (Model::add_y, src/model.rs:188-200) of digit `(y / divisor) % base`
// (or y itself with one digit, or the number y for a regression model).
__global__ __launch_bounds__(256) void k_add_y(int rows, int gb, int e, int max_classes, int digits, int divisor, int base,
                                                const float *__restrict__ y, const float *__restrict__ table,
                                                float *__restrict__ cells) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)gb * rows * e) return;
    const int o = (int)(i % e);
    const size_t r = (i / e) % rows;
    if (max_classes > 0) {
        const int cls = digits > 1 ? ((int)y[r] / divisor) % base : (int)y[r];
        cells[i] += table[(size_t)cls * e + o];
    } else {
        cells[i] += table[o] * y[r] + table[e + o];
    }
}

// h [rows][d] += the in-context stage's target embedding, rounded as Model::add_y rounds it on the host (the product, the
// sum, then the addition to h, none contracted), so that a fit in one call stores the records of the calls apart.
__global__ __launch_bounds__(256) void k_add_y_rows(int rows, int d, int max_classes, const float *__restrict__ y,
                                                    const float *__restrict__ table, float *__restrict__ h) {
#pragma clang fp contract(off)
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)rows * d) return;
    const int o = (int)(i % d);
    const float yr = y[i / d];
    h[i] += max_classes > 0 ? table[(size_t)(int)yr * d + o] : table[o] * yr + table[d + o];
}

__global__ __launch_bounds__(256) void k_scale_by(size_t count, const float *__restrict__ src, float f, float *__restrict__ dst) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) dst[i] = src[i] * f;
}

__global__ __launch_bounds__(256) void k_add_to(size_t count, const float *__restrict__ x, float *__restrict__ sum) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) sum[i] += x[i];
}

// hid [gb * inds][e] += ind [inds][e] (the inducing points' residual, src/fit.rs:388-390)
__global__ __launch_bounds__(256) void k_add_ind(size_t count, int inds, int e, const float *__restrict__ ind,
                                                  float *__restrict__ hid) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) hid[i] += ind[(i / e) % inds * e + i % e];
}

// kv2 [gb * inds][2e] to the column cache: for group g0 + gl, rec = col_kv + (g0 + gl) * gstride + off holds
// K [e][inds] then V [e][inds] (src/fit.rs:394-403).
__global__ __launch_bounds__(256) void k_col_records(int gb, int inds, int e, const float *__restrict__ kv2,
                                                      float *__restrict__ col_kv, size_t gstride, size_t off, int g0) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)gb * 2 * e * inds) return;
    const int k = (int)(i % inds);
    const int j = (int)((i / inds) % (2 * e));
    const int gl = (int)(i / ((size_t)inds * 2 * e));
    col_kv[(size_t)(g0 + gl) * gstride + off + (size_t)j * inds + k] = kv2[((size_t)gl * inds + k) * 2 * e + j];
}

// The inducing points' queries indq [inds][e] over one group's cells, keys and values from kv [gb][rows][2e]; head width
// 16. A workgroup takes one group's head over a range of cells, wavefront w its inducing points 32 w .. of the 128 from
// 128 (blockIdx.z) on: blocks of 128 cells are staged in LDS as split fp16 halves (one block ahead, each thread a key or
// two coordinates of eight values), then attended as in the fused blocks (attend.hpp), the running maximum carried.
// Bound by vector work (about ten instructions a score; of a SIMD's cycles 72% vector, 32% matrix). All heads of a group run on the same XCD, one after another:
// a row's 2 e floats are read 64 bytes a head, and the heads share the lines in that XCD's L2. 100 groups of 10,000
// cells: 518 us a launch, 1,090 on f32 MFMA with 64 cells a step and their loads waited for at each.
constexpr int IND_NT = 128, IND_BUF = IND_NT * 128 + 2 * IND_NT * 32;  // a staged block and its rows of ones
__global__ __launch_bounds__(256, 3) void k_ind_attn16(int gb, int rows, int inds, int e, int heads,
                                                        const float *__restrict__ indq, const float *__restrict__ kv,
                                                        int per_split, float *__restrict__ part_o,
                                                        float *__restrict__ part_ml, float *__restrict__ out) {
    constexpr int NT = IND_NT, STAGED = NT * 128;
    __shared__ __align__(1024) uint8_t lds[2 * IND_BUF];
    __shared__ float red[2][2][2];  // [block parity][keys, values][wavefront of the half]
    __shared__ int shs[2][2];       // [buffer][keys, values]: the staged block's scales
    const int xcd = blockIdx.x & 7, k = blockIdx.x >> 3, h = k % heads, gl = k / heads * 8 + xcd;
    if (gl >= gb) return;
    const int split = blockIdx.y, splits = gridDim.y;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r32 = lane & 31, g = lane >> 5;
    const int qi = blockIdx.z * 128 + wave * 32 + r32, arow = sigma32(r32);
    const bool live = qi < inds;
    const int b0 = split * per_split, nb = min((rows + NT - 1) / NT - b0, per_split);
    const int row0 = b0 * NT;

    // thread t < 128 stages key t, thread 128 + t coordinates 2 (t % 8) and the next of values 8 (t / 8) ..
    const bool st_key = tid < NT;
    const int slot = st_key ? tid : (tid - NT) & ~7, sc2 = 2 * (tid & 7), part = st_key ? 0 : 1;
    // always from the group's own cells (no load behind a branch): past the last cell its again, so that scores need no
    // mask (those values and ones are zero)
    const float *src0 = kv + (size_t)gl * rows * 2 * e + 16 * h + (st_key ? 0 : e + sc2);
    const int per_cell = st_key ? 0 : 1, per_pair = st_key ? 2 : 0;
    float top = 0.0f;
    auto stage_load = [&](int b, float (&stv)[16]) {
        const int at = row0 + b * NT + slot;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float2 v =
                *reinterpret_cast<const float2 *>(src0 + (size_t)min(at + i * per_cell, rows - 1) * 2 * e + i * per_pair);
            stv[2 * i] = v.x;
            stv[2 * i + 1] = v.y;
        }
    };
    auto stage_max = [&](int b, const float (&stv)[16]) {
        float mx = 0.0f;
#pragma unroll
        for (int c = 0; c < 16; c++) mx = fmaxf(mx, fabsf(stv[c]));
        mx = wave_max(mx);
        if (lane == 0) red[b & 1][part][wave & 1] = mx;
    };
    // the scale is that of the largest value so far, so that it only falls from block to block
    auto stage_store = [&](int b, const float (&stv)[16]) {
        const int buf = b & 1;
        top = fmaxf(top, fmaxf(red[buf][part][0], red[buf][part][1]));
        const int s = shift_for_max(top);
        const float f = ldexpf(1.0f, s);
        if ((tid & (NT - 1)) == 0) shs[buf][part] = s;
        uint8_t *const at = lds + buf * IND_BUF;
        const int tg = slot >> 3, left = st_key ? 8 : rows - (row0 + b * NT + slot);  // values of this thread that are there
#pragma unroll
        for (int i = 0; i < 2; i++) {
            float v[8];
#pragma unroll
            for (int t = 0; t < 8; t++) v[t] = st_key ? stv[8 * i + t] : t < left ? stv[2 * t + i] : 0.0f;
            halfx8 hi, lo;
            split8(v, f, hi, lo);
            const int cd = sc2 + i;
            const int place = st_key ? (i * NT + slot) * 16
                                     : NT * 64 + (tg * 16 + (((cd & 3) | ((cd & 4) << 1) | ((cd & 8) >> 1)) ^ (tg & 15))) * 16;
            *reinterpret_cast<halfx8 *>(at + place) = hi;
            *reinterpret_cast<halfx8 *>(at + NT * 32 + place) = lo;
        }
    };
    float st0[16], stv[16];
    stage_load(0, st0);
    if (nb > 1) stage_load(1, stv);
    pad_rows<NT>(lds + STAGED, tid, NT, min(NT, rows - row0));
    pad_rows<NT>(lds + IND_BUF + STAGED, tid, NT, min(NT, rows - row0 - NT));
    // this lane's query, coordinates 8 g .. + 7
    float qv[8], qmax = 0.0f;
    load8(indq + (size_t)(live ? qi : 0) * e + h * 16 + 8 * g, qv);
#pragma unroll
    for (int t = 0; t < 8; t++) qmax = fmaxf(qmax, fabsf(qv[t]));
    const int sq = shift_for_max(half_max(qmax));
    halfx8 qh, ql;
    split8(qv, ldexpf(1.0f, sq), qh, ql);
    stage_max(0, st0);
    if (nb > 1) stage_max(1, stv);
    __syncthreads();
    stage_store(0, st0);

    const bool one = (r32 & 27) == 16;
    const int kb = (g * NT + arow) * 16;
    const int vb = one ? STAGED + 16 * g : NT * 64 + 256 * g + 16 * ((r32 & 15) ^ g);
    float ref = -INFINITY;
    floatx16 o;
#pragma unroll
    for (int v = 0; v < 16; v++) o[v] = 0.0f;
    int sv = 0;
    for (int b = 0; b < nb; b++) {
        const int at = (b & 1) * IND_BUF;
        __syncthreads();  // block b is staged, block b + 1's maxima are in red; everyone is done with block b - 1
        const int sk = shs[b & 1][0], sb = shs[b & 1][1];
        if (b + 1 < nb) {
            stage_store(b + 1, stv);
            // the last block's ones, where it is not whole
            if (rows - row0 - (b + 1) * NT < NT) pad_rows<NT>(lds + (IND_BUF - at) + STAGED, tid, NT, rows - row0 - (b + 1) * NT);
        }
        if (b + 2 < nb) stage_load(b + 2, stv);
        __builtin_amdgcn_sched_barrier(0);  // the loads go out here
        floatx16 sc[4];
#pragma unroll
        for (int j = 0; j < 4; j++) sc[j] = score_tile<NT>(lds + at + kb, j, qh, ql);
        if (b > 0) {
            const float r = ldexpf(1.0f, sb - sv);
#pragma unroll
            for (int t = 0; t < 8; t++) o[t] *= r;
        }
        sv = sb;
        attend_tiles<NT, 4, false>(sc, ldexpf(LOG2E, -(sk + sq)), lds, vb + at, ref, o, [](int) {});
        if (b + 2 < nb) stage_max(b + 2, stv);  // its loads land under the block's attention
    }
    if (!live) return;
    const size_t qr = (size_t)gl * inds + qi;  // the (group, inducing point) item
    float *dst;
    float f;
    if (splits == 1) {
        dst = out + qr * e + h * 16 + 8 * g;
        f = ldexpf(1.0f, -sv) / o[8];
    } else {
        const size_t at = ((size_t)split * gb * inds + qr) * heads + h;
        dst = part_o + at * 16 + 8 * g;
        f = ldexpf(1.0f, -sv);
        if (g == 0) {
            part_ml[at * 2] = ref;
            part_ml[at * 2 + 1] = o[8];
        }
    }
    *reinterpret_cast<float4 *>(dst) = make_float4(o[0] * f, o[1] * f, o[2] * f, o[3] * f);
    *reinterpret_cast<float4 *>(dst + 4) = make_float4(o[4] * f, o[5] * f, o[6] * f, o[7] * f);
}

// The splits of k_ind_attn16 merged: thread t four coordinates of item t / 4 ((group, inducing point, head), 16 floats of
// out in that order; at least one split, every one with keys).
__global__ __launch_bounds__(256) void k_ind_merge(int items, int splits, const float *__restrict__ part_o,
                                                    const float *__restrict__ part_ml, float *__restrict__ out) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x, item = i >> 2;
    if (item >= (size_t)items) return;
    float top = -INFINITY;
    for (int s = 0; s < splits; s++) top = fmaxf(top, part_ml[((size_t)s * items + item) * 2]);
    float l = 0.0f;
    float4 o = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (int s = 0; s < splits; s++) {
        const size_t at = (size_t)s * items + item;
        const float f = exp2_hw(part_ml[at * 2] - top);
        const float4 v = reinterpret_cast<const float4 *>(part_o)[at * 4 + (i & 3)];
        l += part_ml[at * 2 + 1] * f;
        o.x += v.x * f;
        o.y += v.y * f;
        o.z += v.z * f;
        o.w += v.w * f;
    }
    reinterpret_cast<float4 *>(out)[i] = make_float4(o.x / l, o.y / l, o.z / l, o.w / l);
}

// Any head width (the tiny test models): one thread per (group, inducing point, head), streaming over the rows.
__global__ __launch_bounds__(256) void k_ind_attn_plain(int gb, int rows, int inds, int e, int heads,
                                                         const float *__restrict__ indq, const float *__restrict__ kv,
                                                         float *__restrict__ out) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)gb * inds * heads) return;
    const int h = (int)(i % heads), qi = (int)((i / heads) % inds), gl = (int)(i / ((size_t)heads * inds));
    const int hd = e / heads;
    const float *qr = indq + (size_t)qi * e + h * hd;
    const float *base = kv + (size_t)gl * rows * 2 * e;
    float *o = out + ((size_t)gl * inds + qi) * e + h * hd;
    float m = -INFINITY, l = 0.0f;
    for (int c = 0; c < hd; c++) o[c] = 0.0f;
    for (int r = 0; r < rows; r++) {
        const float *row = base + (size_t)r * 2 * e;
        float s = 0.0f;
        for (int c = 0; c < hd; c++) s += qr[c] * row[h * hd + c];
        const float mnew = fmaxf(m, s);
        const float alpha = fast_exp(m - mnew), p = fast_exp(s - mnew);
        l = l * alpha + p;
        for (int c = 0; c < hd; c++) o[c] = o[c] * alpha + p * row[e + h * hd + c];
        m = mnew;
    }
    for (int c = 0; c < hd; c++) o[c] /= l;
}

// tok [rb][T][e]: class tokens then cells of rows r0.. from emb [features][rows][e]. A workgroup per row, 16 bytes a
// thread (e a multiple of 4).
__global__ __launch_bounds__(256) void k_tokens_gmajor(int rb, int r0, int rows, int cls, int features, int e,
                                                        const float *__restrict__ cls_tokens,
                                                        const float *__restrict__ emb, float *__restrict__ tok) {
    const int r = blockIdx.x;
    if (r >= rb) return;
    const int e4 = e / 4, T = cls + features;
    float4 *dst = reinterpret_cast<float4 *>(tok + (size_t)r * T * e);
    for (int i = threadIdx.x; i < T * e4; i += 256) {
        const int t = i / e4, o = i - t * e4;
        const float4 *src = t < cls ? reinterpret_cast<const float4 *>(cls_tokens + (size_t)t * e)
                                    : reinterpret_cast<const float4 *>(emb + ((size_t)(t - cls) * rows + r0 + r) * e);
        dst[i] = src[o];
    }
}

// Cells of e floats between [rows][g][e] and [g][rows][e]: e / 4 threads a cell, 16 bytes each (e a multiple of 4).
__global__ __launch_bounds__(256) void k_regroup(int rows, int g, int e, const float *__restrict__ src,
                                                  float *__restrict__ dst, bool to_gmajor) {
    const int e4 = e / 4, per = 256 / e4;
    const int slot = threadIdx.x / e4, o = threadIdx.x - slot * e4;
    const long cell = (long)blockIdx.x * per + slot;  // in the destination's order
    if (slot >= per || cell >= (long)rows * g) return;
    long from;
    if (to_gmajor) {
        const long gi = cell / rows, r = cell - gi * rows;
        from = r * g + gi;
    } else {
        const long r = cell / g, gi = cell - r * g;
        from = gi * rows + r;
    }
    reinterpret_cast<float4 *>(dst)[cell * e4 + o] = reinterpret_cast<const float4 *>(src)[from * e4 + o];
}

// ---- launchers ---------------------------------------------------------------------------------------------
void fit_cells(hipStream_t s, const tah_weights *w, const float *x, int rows, int features, int g0, int gb, float *cells,
               const float *y) {
    if (w->group > 8 || w->group < 1) throw ArgError{"column stage: feature group size must be 1..8"};
    if (w->e % 4) throw ArgError{"column stage: embedding width must be a multiple of 4"};
    for (int k = 0; k < gb; k += 65535) {  // a launch's groups
        const dim3 grid((rows + FIT_ROWS - 1) / FIT_ROWS, std::min(gb - k, 65535));
        float *at = cells + (size_t)k * rows * w->e;
        if (w->group == 3)
            hipLaunchKernelGGL(k_fit_cells<3>, grid, dim3(256), 0, s, rows, features, g0 + k, 3, w->e, x, w->in_w, w->in_b, y,
                               w->max_classes, w->col_y, at);
        else
            hipLaunchKernelGGL(k_fit_cells<0>, grid, dim3(256), 0, s, rows, features, g0 + k, w->group, w->e, x, w->in_w,
                               w->in_b, y, w->max_classes, w->col_y, at);
    }
    TAH_LAUNCHED();
}

void add_y_cells(hipStream_t s, const tah_weights *w, const float *y, int rows, int gb, int digits, int divisor, int base,
                 float *cells) {
    const size_t count = (size_t)gb * rows * w->e;
    hipLaunchKernelGGL(k_add_y, blocks_of(count), dim3(256), 0, s, rows, gb, w->e, w->max_classes, digits, divisor, base, y,
                       w->col_y, cells);
    TAH_LAUNCHED();
}

// rows [rows][d] += the in-context stage's target embedding (Model::add_y, src/model.rs:188-200).
void add_y_rows(hipStream_t s, const tah_weights *w, const float *y, int rows, float *h) {
    hipLaunchKernelGGL(k_add_y_rows, blocks_of((size_t)rows * w->d), dim3(256), 0, s, rows, w->d, w->max_classes, y, w->icl_y,
                       h);
    TAH_LAUNCHED();
}

void scale_by(hipStream_t s, size_t count, const float *src, float f, float *dst) {
    hipLaunchKernelGGL(k_scale_by, blocks_of(count), dim3(256), 0, s, count, src, f, dst);
    TAH_LAUNCHED();
}

void add_to(hipStream_t s, size_t count, const float *x, float *sum) {
    hipLaunchKernelGGL(k_add_to, blocks_of(count), dim3(256), 0, s, count, x, sum);
    TAH_LAUNCHED();
}

void add_ind(hipStream_t s, size_t count, int inds, int e, const float *ind, float *hid) {
    hipLaunchKernelGGL(k_add_ind, blocks_of(count), dim3(256), 0, s, count, inds, e, ind, hid);
    TAH_LAUNCHED();
}

void col_records(hipStream_t s, int gb, int inds, int e, const float *kv2, float *col_kv, size_t gstride, size_t off, int g0) {
    const size_t count = (size_t)gb * 2 * e * inds;
    hipLaunchKernelGGL(k_col_records, blocks_of(count), dim3(256), 0, s, gb, inds, e, kv2, col_kv, gstride, off, g0);
    TAH_LAUNCHED();
}

void regroup(hipStream_t s, int rows, int g, int e, const float *src, float *dst, bool to_group_major) {
    if (e % 4 || e > 1024) throw ArgError{"regroup: cell width must be a multiple of 4, at most 1024"};
    const size_t per = 256 / (e / 4);
    hipLaunchKernelGGL(k_regroup, dim3((unsigned)(((size_t)rows * g + per - 1) / per)), dim3(256), 0, s, rows, g, e, src,
                       dst, to_group_major);
    TAH_LAUNCHED();
}

void tokens_gmajor(hipStream_t s, const tah_weights *w, int rb, int r0, int rows, int features, const float *emb, float *tok) {
    if (w->e % 4) throw ArgError{"row stage: embedding width must be a multiple of 4"};
    hipLaunchKernelGGL(k_tokens_gmajor, dim3(rb), dim3(256), 0, s, rb, r0, rows, w->cls, features, w->e, w->cls_tokens,
                       emb, tok);
    TAH_LAUNCHED();
}

// Ranges of cells a group's head is split into, in blocks of 128: about 4,096 workgroups in all (768 run at once), at
// least two blocks each. A launch with its merge, us, with 1,024, 2,048, 4,096 and 8,192 workgroups instead: 100 groups
// of 10,000 cells 601, 522, 516, 518; 200 of 1,500 157, 158, 164, 162; 20 of 3,000 43, 46, 48, 46; 12 of 400 13 to 14.
static int ind_splits(const tah_weights *w, int rows, int gb) {
    const int blocks = (rows + IND_NT - 1) / IND_NT;
    const int tiles = gb * w->col_heads * ((w->inds + 127) / 128);
    const int want = std::min(std::max(1, 4096 / std::max(1, tiles)), std::max(1, blocks / 2));
    const int per = (blocks + want - 1) / want;
    return (blocks + per - 1) / per;
}

static bool ind_mfma(const tah_weights *w) { return w->e / w->col_heads == 16 && w->inds % 64 == 0; }

size_t ind_attention_work_bytes(const tah_weights *w, int rows, int gb) {
    if (!ind_mfma(w)) return 0;
    const int splits = ind_splits(w, rows, gb);
    if (splits == 1) return 0;
    return sizeof(float) * (size_t)splits * gb * w->inds * w->col_heads * (w->e / w->col_heads + 2) + 256;
}

// The inducing points' queries indq [inds][e] over each of gb groups' cells (kv [gb][rows][2e]) to out
// [gb * inds][e], normalised.
void ind_attention(hipStream_t s, const tah_weights *w, int rows, int gb, const float *indq, const float *kv, float *out,
                   void *work) {
    const int e = w->e, heads = w->col_heads, inds = w->inds;
    if (!ind_mfma(w)) {
        hipLaunchKernelGGL(k_ind_attn_plain, blocks_of((size_t)gb * inds * heads), dim3(256), 0, s, gb, rows, inds, e, heads,
                           indq, kv, out);
        TAH_LAUNCHED();
        return;
    }
    const int splits = ind_splits(w, rows, gb);
    const int per = ((rows + IND_NT - 1) / IND_NT + splits - 1) / splits;
    float *part_o = splits > 1 ? static_cast<float *>(work) : nullptr;
    float *part_ml = splits > 1 ? part_o + (size_t)splits * gb * inds * heads * (e / heads) : nullptr;
    const dim3 grid((gb + 7) / 8 * 8 * heads, splits, (inds + 127) / 128);
    hipLaunchKernelGGL(k_ind_attn16, grid, dim3(256), 0, s, gb, rows, inds, e, heads, indq, kv, per, part_o, part_ml, out);
    TAH_LAUNCHED();
    if (splits > 1) {
        const int items = gb * inds * heads;
        hipLaunchKernelGGL(k_ind_merge, blocks_of((size_t)items * 4), dim3(256), 0, s, items, splits, part_o, part_ml, out);
        TAH_LAUNCHED();
    }
}

}  // namespace tah
