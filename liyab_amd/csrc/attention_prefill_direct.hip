// Causal attention of prompt portions over paged bfloat16 keys and values for heads of 64 and of 128: what
// attention_prefill.hip computes (see its head: transposed scores, a query's scores in one lane and the lane 32 apart, a lagging
// reference for the exponentials, 32-bit maximum, exponentials, sums and outputs), with the keys and values straight from their
// pages into LDS (global_load_lds, 16 bytes a lane).
//
// What bounds it: a wave's 32 queries and 64 keys take 512 cycles of the matrix cores at 64 a head, and some 150 vector instructions (a
// maximum, a multiply-add, an exponential, a sum and half a conversion a score), which overlap only across the waves of a SIMD. The kernel
// that keeps a ring of keys in registers needs 312 of them: one wave a SIMD, its chain of products, maximum, exponentials and products laid bare.
// Without the ring heads of 64 take 166 a wave of two streams and 112 to 123 of one, three and four waves a SIMD; 173 to 176 where a lane finds its own row, 215 to
// 223 with scores to work on (two waves; one stream 122 to 162), and heads of 128 173 to 230 (two waves). A load's rows come from one page
// where pages allow it, so that its address is a scalar: a lookup a lane cost 60 vector instructions a step. The sums are in the other
// kernel's order (blocks of 32 keys, as many streams, the same merges): the same bits.
// us a layer, before and now: 1 x 8,001 tokens, 12 heads 166 -> 143 (0.69 PFLOP/s; in a pass, between the products, 180 -> 150), 8 x 992 of 25 heads 65 -> 44.4 (71 -> 48), 2 x 1,024 of 12 heads 19.2 -> 16.0,
// 4 x 192 behind 256 of 16 heads 11.7 -> 8.4, 8 x 1,000 of 12 heads of 128 81 -> 52; with a sink 4 x 410 of 12 heads 18.9 -> 10.1.
// The row table takes a word a page of the block tables' width, so that three workgroups of 128 queries share a compute unit's LDS up to 1,365 pages; with
// 2,048 there are two (8 x 992 49.6, 1 x 8,001 138).
// Measured and left: one stream of 64 keys (7, 2 and 5 % faster for the first three: other roundings), two stages or four in place of three,
// an order of the tiles that deals the long ones out from both ends (no faster).
#include "attention_prefill.h"
#include "attention_prefill_walk.h"
#include "common.h"
#include "launchers.h"

namespace liyab {

template <int HD, int QG, int KS, int NS, int STAGES, int MIN_WAVES, bool SCORED, bool BY_LOAD>
__global__ void __launch_bounds__(64 * QG * KS, MIN_WAVES)
attention_prefill_direct_kernel(PrefillArgs p, int page_shift) {
    // heads vary fastest: the work list has the longest tiles first, and workgroups start in the
    // grid's order, so that every head's longest tile starts before anybody's short one
    attention_prefill_walk<HD, QG, KS, NS, STAGES, SCORED, BY_LOAD>(p, page_shift, blockIdx.x, blockIdx.y);
}

template <int HD, int QG, int KS, int NS, int STAGES, int MIN_WAVES, bool SCORED, bool BY_LOAD>
int launch_direct_pages(const PrefillArgs& p, int n_tiles, int page_shift, hipStream_t stream) {
    typedef DirectShape<HD, QG, KS, NS, STAGES> S;
    auto kern = attention_prefill_direct_kernel<HD, QG, KS, NS, STAGES, MIN_WAVES, SCORED, BY_LOAD>;
    constexpr int most = static_cast<int>(S::BYTES) + kPrefillMaxBlocks * 4;
    static_assert(most <= 160 * 1024, "a workgroup's LDS");
    static bool ready = false;  // once per instantiation, outside any stream capture's first use
    if (!ready) {
        hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, most);
        ready = true;
    }
    kern<<<dim3(p.n_head, n_tiles), S::THREADS, S::BYTES + static_cast<size_t>(p.max_blocks) * 4, stream>>>(p, page_shift);
    return check_launch("attention_prefill");
}

template <int HD, int QG, int KS, int NS, int STAGES, int MIN_WAVES, bool SCORED>
int launch_direct_as(const PrefillArgs& p, int n_tiles, int page_shift, hipStream_t stream) {
    // Two streams and a row a lane to find do not fit the registers of three waves a SIMD (9 spilled, 40 bytes of scratch a lane, read back every step): two
    // waves (8,001 tokens of 12 heads in pages of 24 178 -> 154 us, of 4 173 -> 145; 2 x 1,024 of 25 heads 27.3 -> 22.9 and 26.8 -> 21.9).
    const bool by_load = page_shift >= 0 && p.page_size * HD >= 512 && !(SCORED && p.window > 0 && p.keep_first > 0);
    return by_load ? launch_direct_pages<HD, QG, KS, NS, STAGES, MIN_WAVES, SCORED, true>(p, n_tiles, page_shift, stream)
                   : launch_direct_pages<HD, QG, KS, NS, STAGES, NS == 2 ? 2 : MIN_WAVES, SCORED, false>(p, n_tiles, page_shift, stream);
}

template <bool SCORED>
int launch_prefill_direct(const PrefillArgs& p, int n_tiles, int tile, int ksplit, int page_shift, hipStream_t stream) {
    // two streams a wave where tiles of 128 queries leave it the registers
#define LIYAB_DIRECT(HD, QG, KS, STAGES, MIN_WAVES) \
    launch_direct_as<HD, QG, KS, (HD == 64 && QG == 4) ? 2 : 1, STAGES, SCORED ? 2 : MIN_WAVES, SCORED>(p, n_tiles, page_shift, stream)
    if (p.hd == 64) {
        if (tile == 128) return ksplit == 1 ? LIYAB_DIRECT(64, 4, 1, 3, 3) : LIYAB_DIRECT(64, 4, 2, 2, 2);
        if (ksplit == 1) return LIYAB_DIRECT(64, 2, 1, 3, 3);
        return ksplit == 2 ? LIYAB_DIRECT(64, 2, 2, 3, 3) : LIYAB_DIRECT(64, 2, 4, 2, 2);
    }
    if (tile == 128) return ksplit == 1 ? LIYAB_DIRECT(128, 4, 1, 3, 2) : LIYAB_DIRECT(128, 4, 2, 2, 2);
    return ksplit == 1 ? LIYAB_DIRECT(128, 2, 1, 3, 2) : LIYAB_DIRECT(128, 2, 2, 3, 2);
#undef LIYAB_DIRECT
}
template int launch_prefill_direct<false>(const PrefillArgs&, int, int, int, int, hipStream_t);
template int launch_prefill_direct<true>(const PrefillArgs&, int, int, int, int, hipStream_t);

}  // namespace liyab
