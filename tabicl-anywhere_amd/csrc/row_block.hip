// Launches of the row stage's fused block (row_block.hpp).
#include "row_block.hpp"

namespace tah {

extern template void launch_row_next<4, 2, 1>(const RowLaunch &);
extern template void launch_row_next<4, 2, 2>(const RowLaunch &);
extern template void launch_row_next<4, 1, 3>(const RowLaunch &);
extern template void launch_row_next<4, 1, 4>(const RowLaunch &);
extern template void launch_row_next<8, 1, 5>(const RowLaunch &);
extern template void launch_row_next<8, 1, 6>(const RowLaunch &);
extern template void launch_row_next<8, 1, 7>(const RowLaunch &);
extern template void launch_row_next<8, 1, 8>(const RowLaunch &);

// Without the next block's keys and values; FF: with the feed-forward half.
template <bool FF, int W, int R, int NTL>
static void launch_row_last(const RowLaunch &a) {
    const DevBlock &b = a.b;
    hipLaunchKernelGGL((k_row_block<FF, false, W, R, NTL>), dim3((a.n + R - 1) / R), dim3(64 * W), 0, a.s, a.n, a.T, a.T,
                       a.tok, a.kv, a.cosv, a.sinv, b.n1w, b.n1b, b.inimg, b.ins, b.in_b, b.outimg, b.outs, b.out_b,
                       FF ? b.n2w : nullptr, FF ? b.n2b : nullptr, FF ? b.l1img : nullptr, FF ? b.l1b : nullptr,
                       FF ? b.l1s : 0, FF ? b.l2img : nullptr, FF ? b.l2b : nullptr, FF ? b.l2s : 0, KvNext{});
}

bool row_block_fits(const DevBlock &b, int T) {
    return b.d == 128 && b.heads == 8 && b.inimg && b.outimg && T >= 1 && T <= 256;
}

void row_block(hipStream_t s, int n, int T, float *tok, const float *kv, const float *cosv, const float *sinv,
               const DevBlock &b, bool ff, const DevBlock *next, float *kv_next, int keep) {
    if (n <= 0) return;
    if (!row_block_fits(b, T) || (reinterpret_cast<uintptr_t>(tok) & 15) || (reinterpret_cast<uintptr_t>(kv) & 15))
        throw ArgError{"row_block: needs e = 128, 8 heads, weight images, at most 256 tokens and aligned rows"};
    if (ff && !block_ff_fits(b)) throw ArgError{"row_block: no fused feed-forward weights for this shape"};
    if (next && (!ff || !row_kv_fits(*next) || !kv_next || (reinterpret_cast<uintptr_t>(kv_next) & 15)))
        throw ArgError{"row_block: the next block's keys and values need the fused feed-forward, e = 128, its "
                       "projection image and an aligned destination"};
    if (keep < 0) keep = T;
    if (keep > T || (keep < T && !next))
        throw ArgError{"row_block: only a block that forms the next one's keys and values may leave tokens unwritten"};
    const KvNext kn = next ? KvNext{next->inimg + (size_t)128 * 128 * 4, next->ins, next->n1w, next->n1b,
                                    next->in_b + 128, kv_next}
                           : KvNext{};
    const RowLaunch a{s, n, T, keep, tok, kv, cosv, sinv, b, kn};
    // by the row's tokens in tiles of 32: up to two tiles two rows share a workgroup of four wavefronts (a row of its own
    // would leave half of them without tokens), up to four tiles one row takes it, past that eight wavefronts
    const int tiles = (T + 31) / 32;
    if (next) {
        switch (tiles) {
            case 1: launch_row_next<4, 2, 1>(a); break;
            case 2: launch_row_next<4, 2, 2>(a); break;
            case 3: launch_row_next<4, 1, 3>(a); break;
            case 4: launch_row_next<4, 1, 4>(a); break;
            case 5: launch_row_next<8, 1, 5>(a); break;
            case 6: launch_row_next<8, 1, 6>(a); break;
            case 7: launch_row_next<8, 1, 7>(a); break;
            default: launch_row_next<8, 1, 8>(a); break;
        }
    } else if (ff) {  // the few-row paths' last whole block: fewer kernels, the tile count rounded up
        if (tiles <= 1) launch_row_last<true, 4, 2, 1>(a);
        else if (tiles <= 2) launch_row_last<true, 4, 2, 2>(a);
        else if (tiles <= 4) launch_row_last<true, 4, 1, 4>(a);
        else launch_row_last<true, 8, 1, 8>(a);
    } else {
        if (tiles <= 2) launch_row_last<false, 4, 2, 2>(a);
        else if (tiles <= 4) launch_row_last<false, 4, 1, 4>(a);
        else launch_row_last<false, 8, 1, 8>(a);
    }
    TAH_LAUNCHED();
}

}  // namespace tah
