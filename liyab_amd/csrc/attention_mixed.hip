// Attention of a step that has both prompt portions and tokens taken one at a time, heads of 64, in one launch: a workgroup is a tile of a portion's queries
// (attention_prefill_walk.h) or one token's head (attention_decode_walk.h), with the bits that each has in a kernel of its own.
// What bounds either is its longest walk over the keys while half of the chip's places stand empty (medium's sizes, 12 tokens and 4 portions of some 190: 192 workgroups of 12.1 us, then
// some 200 of 9.6): side by side they take little more than the longer one, and a link of the step's chain goes. The step 2,101 -> 1,905 us, 8 us a layer;
// ones of small's sizes with few single tokens, whose keys are cut, 1,167 -> 975, 1,404 -> 1,284, 1,455 -> 1,265, with more 860 -> 772. Single tokens first: theirs are the longer walks. Their sums lie in the tiles' ring, so that two workgroups share a
// compute unit's LDS as before.
#include "attention_decode_walk.h"
#include "attention_prefill_walk.h"
#include "common.h"
#include "launchers.h"

namespace liyab {

struct MixedArgs {
    const int *tok_list, *tok_seq, *tok_pos;
    float* partials;
    int n, n_tiles, n_splits, heads_first;
};

// QG, KS, NS, STAGES: as attention_prefill_direct_kernel's; DW: waves a single token's head, or split of its keys, takes. A workgroup has as many as the larger of the two, the
// others leave at once (a barrier counts the waves that are there). MIN_WAVES a SIMD: the workgroups that LDS lets a compute unit hold.
template <int QG, int KS, int NS, int STAGES, int DW, int MIN_WAVES>
__global__ void __launch_bounds__(64 * (QG * KS > DW ? QG * KS : DW), MIN_WAVES)
attention_mixed_kernel(PrefillArgs p, MixedArgs d, int page_shift) {
    extern __shared__ __attribute__((aligned(1024))) bf16_t ring[];
    const int pairs = d.n * p.n_head, singles = pairs * d.n_splits, block = blockIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    if (block < singles) {
        if (wave >= DW) return;
        const int z = block / pairs, at = block - z * pairs, slot = d.heads_first ? at / p.n_head : at % d.n, h = d.heads_first ? at % p.n_head : at / d.n;
        attention_decode_walk<bf16_t, 8, DW, 4, false, DW == 4>(*reinterpret_cast<DecodeLds<8, DW>*>(ring), slot, h, z, p.out, p.out_stride, p.q, p.q_stride, p.kc, p.vc,
                                                               p.block_tables, p.max_blocks, d.tok_list, d.tok_seq, d.tok_pos, p.scale, p.window, p.n_head, p.n_kv_head, 64,
                                                               p.page_size, page_shift, 0, d.n_splits, 31 - __builtin_clz(d.n_splits), 0, d.partials, p.num_pages, 0.0f, nullptr,
                                                               0, nullptr, 0);
    } else {
        if (wave >= QG * KS) return;
        const int t = block - singles;
        attention_prefill_walk<64, QG, KS, NS, STAGES, false, true>(p, page_shift, t % p.n_head, t / p.n_head);
    }
}

template <int QG, int KS, int NS, int STAGES, int DW, int MIN_WAVES>
int launch_mixed(const PrefillArgs& p, const MixedArgs& d, int page_shift, hipStream_t stream) {
    typedef DirectShape<64, QG, KS, NS, STAGES> S;
    auto kern = attention_mixed_kernel<QG, KS, NS, STAGES, DW, MIN_WAVES>;
    constexpr int most = static_cast<int>(S::BYTES) + kPrefillMaxBlocks * 4, waves = QG * KS > DW ? QG * KS : DW;
    static_assert(most <= 160 * 1024 && sizeof(DecodeLds<8, DW>) <= S::BYTES, "a workgroup's LDS");
    static bool ready = false;  // once per instantiation, outside any stream capture's first use
    if (!ready) {
        hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, most);
        ready = true;
    }
    kern<<<(d.n * d.n_splits + d.n_tiles) * p.n_head, 64 * waves, S::BYTES + static_cast<size_t>(p.max_blocks) * 4, stream>>>(p, d, page_shift);
    if (const int rc = check_launch("attention_mixed")) return rc;
    return d.n_splits > 1 ? merge_decode_splits(p.out, p.out_stride, d.tok_list, d.partials, d.n, p.n_head, 64, d.n_splits, stream) : 0;
}

}  // namespace liyab

using namespace liyab;

// liyab_attention_prefill (bfloat16, heads of 64, pages a power of two of 8 positions or more) and, for the rows tok_list[0..n), liyab_attention_decode in n_splits
// (a power of two; more than one: merged behind it, `partials` as there) on `waves` waves: 4 or 8 beside tiles of 64 with 2 or 4 waves a query group, 4 beside tiles of 128 with one.
// The rows of both are written once each.
extern "C" int liyab_attention_mixed(void* out, int64_t out_stride, const void* q, int64_t q_stride, const void* kc, const void* vc, const int* block_tables,
                                     int max_blocks, const int* work, int n_tiles, int tile, int ksplit, const int* tok_list, const int* tok_seq, const int* tok_pos,
                                     int n, int n_splits, int waves, float* partials, float scale, int window, int n_head, int n_kv_head, int page_size, int num_pages,
                                     hipStream_t stream) {
    LIYAB_REQUIRE(out && q && kc && vc && block_tables && work && tok_list && tok_seq && tok_pos, "attention_mixed: null pointer");
    LIYAB_REQUIRE(n >= 1 && n_tiles >= 1 && n_head > 0 && n_kv_head > 0 && n_head % n_kv_head == 0 && max_blocks > 0 && max_blocks <= AD_MAX_BLOCKS && max_blocks <= kPrefillMaxBlocks,
                  "attention_mixed: bad sizes (%d tokens, %d tiles, %d of %d heads, %d pages a request)", n, n_tiles, n_head, n_kv_head, max_blocks);
    LIYAB_REQUIRE(n_splits >= 1 && n_splits <= 64 && (n_splits & (n_splits - 1)) == 0 && (n_splits == 1 || partials != nullptr), "attention_mixed: bad split count %d", n_splits);
    LIYAB_REQUIRE((static_cast<int64_t>(n) * n_splits + n_tiles) * n_head <= INT_MAX, "attention_mixed: %d tokens and %d tiles of %d heads", n, n_tiles, n_head);
    LIYAB_REQUIRE(page_size >= 8 && (page_size & (page_size - 1)) == 0 && num_pages > 0, "attention_mixed: pages of %d positions are no power of two from 8 on", page_size);
    LIYAB_REQUIRE(static_cast<int64_t>(num_pages) * n_kv_head * page_size <= UINT32_MAX, "attention_mixed: caches of %d pages hold too many rows", num_pages);
    auto al16 = [](const void* x) { return (reinterpret_cast<uintptr_t>(x) & 15) == 0; };
    LIYAB_REQUIRE(al16(out) && al16(q) && al16(kc) && al16(vc) && q_stride % 8 == 0 && out_stride % 8 == 0, "attention_mixed: rows must be 16-byte aligned");
    LIYAB_REQUIRE(q_stride >= static_cast<int64_t>(n_head) * 64 && out_stride >= static_cast<int64_t>(n_head) * 64, "attention_mixed: row strides are shorter than heads x 64");
    LIYAB_REQUIRE(scale > 0.0f && window >= 0, "attention_mixed: a scale of %g or a window of %d", scale, window);
    const PrefillArgs p{static_cast<bf16_t*>(out), out_stride, static_cast<const bf16_t*>(q), q_stride, static_cast<const bf16_t*>(kc), static_cast<const bf16_t*>(vc),
                        block_tables, max_blocks, work, scale, window, n_head, n_kv_head, 64, page_size, num_pages, 0.0f, nullptr, 0, nullptr, 0};
    const MixedArgs d{tok_list, tok_seq, tok_pos, partials, n, n_tiles, n_splits, n_head == n_kv_head ? 1 : 0};
    const int page_shift = __builtin_ctz(page_size);
    if (tile == 64 && ksplit == 2 && waves == 4) return launch_mixed<2, 2, 1, 3, 4, 3>(p, d, page_shift, stream);
    if (tile == 64 && ksplit == 2 && waves == 8) return launch_mixed<2, 2, 1, 3, 8, 4>(p, d, page_shift, stream);
    if (tile == 64 && ksplit == 4 && waves == 4) return launch_mixed<2, 4, 1, 2, 4, 4>(p, d, page_shift, stream);
    if (tile == 64 && ksplit == 4 && waves == 8) return launch_mixed<2, 4, 1, 2, 8, 4>(p, d, page_shift, stream);
    if (tile == 128 && ksplit == 1 && waves == 4) return launch_mixed<4, 1, 2, 3, 4, 3>(p, d, page_shift, stream);
    return fail(1, "attention_mixed: tiles of %d queries with %d waves a query group beside tokens on %d are not taken", tile, ksplit, waves);
}
