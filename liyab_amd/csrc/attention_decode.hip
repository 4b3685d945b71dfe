// Attention for tokens taken one at a time (decoding, short prompt portions)
// over paged keys and values (bfloat16, or 32-bit for the 32-bit path), with
// the keys of a token cut into splits so that few tokens still fill the chip.
//
// Grid (token, query head, split). A workgroup of 4, 8 or 16 waves walks its split's
// keys; LPK lanes share a key (each holds 8 consecutive dimensions, 16
// bytes), so a wave takes 64 / LPK keys a pass, read straight from the pages
// through the block table. Each lane group keeps a running maximum, sum and
// weighted values (the reference's per-span partial softmax,
// src/core/transformer.cpp:2327-2358); groups, then waves, then splits are
// merged in a fixed order by rescaling to the common maximum (:2367-2385).
// With `chunk` keys a split (instead of the token's keys divided by the number of
// splits) and four waves, which lane adds which key and which sums are merged
// follow from the token's position alone, as the reference cuts (:2136-2139):
// the form of the 32-bit path and of the batch-invariant mode.
// What bounds it: with many pairs the caches' reads (64 tokens of 25 heads over 256 to 1,015 keys, 261 MB: 50.3 us, where reading the same bytes
// and doing nothing takes 45.5), so four waves ask for the next trip's keys and values before they absorb the ones they have, where that pays
// (next_trip_ahead_pays); eight and sixteen hold as much in flight by their number (24 tokens of 12 heads on eight: 12.7, 13.1 with the next trip's
// loads in flight, whose registers cost a workgroup a compute unit). With few pairs the instructions around the loads: only a wave's last trip looks at which
// keys it has, and the other trips and both forms' loads are free of branches. us, with every key looked at and nothing asked for ahead / now, caches not
// read before, heads of 64: 64 tokens of 25 heads 51.7 / 50.3, 32 of 16 over 100 to 900 keys 21.5 / 17.2, 17 of 12 over 200 to 1,000 on eight waves 14.5 / 13.1,
// one of 12 at 1,024 in 8 splits 5.2 / 4.8.
// The reference cuts a token's keys by its position only (:2136-2139,
// 2225-2227) to keep bits equal; here the number of splits follows the batch
// (more splits when few tokens are in flight), which moves results by
// rounding only. Scores, exponentials and sums are 32-bit.
#include "attention_decode_walk.h"
#include "common.h"
#include "launchers.h"

namespace liyab {

template <typename T, int LPK, int AD_WAVES, int AD_U, bool SCORED, bool AHEAD>
__global__ void __launch_bounds__(64 * AD_WAVES)
attention_decode_kernel(T* __restrict__ out, int64_t out_stride, const T* __restrict__ q, int64_t q_stride,
                        const T* __restrict__ kc, const T* __restrict__ vc,
                        const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ tok_list,
                        const int* __restrict__ tok_seq, const int* __restrict__ tok_pos, float scale, int window,
                        int n_head, int n_kv_head, int hd, int page_size, int page_shift, int rows_are_requests,
                        int n_splits, int split_shift, int chunk, float* __restrict__ partials, int num_pages, int heads_first, float softcap = 0.0f,
                        const float* __restrict__ bias_table = nullptr, int max_dist = 0, const float* __restrict__ sinks = nullptr,
                        int keep_first = 0) {
    __shared__ DecodeLds<LPK, AD_WAVES> shared;
    // (which of the two the grid runs along first: heads_first_pays)
    attention_decode_walk<T, LPK, AD_WAVES, AD_U, SCORED, AHEAD>(shared, heads_first ? blockIdx.y : blockIdx.x, heads_first ? blockIdx.x : blockIdx.y, blockIdx.z,
                                                                 out, out_stride, q, q_stride, kc, vc, block_tables, max_blocks, tok_list, tok_seq, tok_pos, scale, window, n_head, n_kv_head, hd, page_size, page_shift,
                                                                rows_are_requests, n_splits, split_shift, chunk, partials, num_pages, softcap, bias_table, max_dist, sinks, keep_first);
}

// Splits of a (token, head) merged in split order (the same operations as the end of the kernel above).
template <typename T>
__global__ void attention_merge_kernel(T* __restrict__ out, int64_t out_stride, const int* __restrict__ tok_list,
                                       const float* __restrict__ partials, int n_head, int hd, int n_splits,
                                       const float* __restrict__ sinks = nullptr) {
    // The splits' maxima and sums go to LDS first, a lane a split, and the values are fetched
    // eight splits at a time before they are used: the sums below are one chain in split order,
    // and a load at a time inside it would cost its latency once a split.
    __shared__ float sm[64], sl[64];
    const int slot = blockIdx.x, h = blockIdx.y, e = threadIdx.x;
    const int t = tok_list != nullptr ? tok_list[slot] : slot;
    const float* p = partials + (static_cast<int64_t>(slot) * n_head + h) * n_splits * (hd + 4);
    const int ec = min(e, hd - 1);
    float a[8];  // the first eight splits' values are on their way while the maxima and sums go through LDS
#pragma unroll
    for (int u = 0; u < 8; ++u) a[u] = p[min(u, n_splits - 1) * (hd + 4) + ec];
    for (int z = e; z < n_splits; z += blockDim.x) {
        sm[z] = p[z * (hd + 4) + hd];
        sl[z] = p[z * (hd + 4) + hd + 1];
    }
    __syncthreads();
    if (e >= hd) return;
    float M = -INFINITY;
    for (int z = 0; z < n_splits; ++z) M = fmaxf(M, sm[z]);
    float sum = 0.0f, o = 0.0f;
    for (int z0 = 0; z0 < n_splits; z0 += 8) {
        if (z0 > 0) {
#pragma unroll
            for (int u = 0; u < 8; ++u) a[u] = p[min(z0 + u, n_splits - 1) * (hd + 4) + e];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            if (z0 + u >= n_splits) break;
            const float m = sm[z0 + u];
            if (m == -INFINITY) continue;
            const float w = exp_for<T>(m - M);
            sum = fmaf(w, sl[z0 + u], sum);
            o = fmaf(w, a[u], o);
        }
    }
    if (sinks != nullptr) {
        float one[1] = {o};
        add_sink<T, 1>(M, sum, one, sinks[h]);
        o = one[0];
    }
    out[static_cast<int64_t>(t) * out_stride + static_cast<int64_t>(h) * hd + e] = from_float<T>(o / sum);
}

// Whether the grid runs along the heads first. Workgroups go to the 8 XCDs in turn, each with 4 MB of L2. With tokens first, and a
// number of tokens that 8 divides, an XCD has all of a token, and the one with the long contexts is waited for; with heads first a
// token's heads spread over the XCDs. Measured, us a call, tokens first -> heads first; 64 wide heads, contexts of 256 to 1,015 keys:
//   one token a request: 64 tokens of 25 heads 58.8 -> 54.6, of 16 heads 36.9 -> 34.7, 128 of 12 heads 53.9 -> 50.8; splits left to the
//     projection, 1 to 16 tokens, 1-6 % less; up to 16 tokens uncut or merged here: even, scored (8 tokens, a window of 512) 7.4 -> 7.8;
//   short portions (up to 8 tokens a request, side by side: their common keys stay in an XCD's L2): 8 x 8 tokens of 12 heads
//     22.5 -> 16.2, 32 x 8 of 20 heads 122 -> 64, of 25 heads even;
//   whole prompts in fixed chunks (neighbours read the same keys): heads first while the keys and values of the heads that fall
//     to one XCD, n_head / gcd(n_head, 8) of them, stay in its L2: 300 rows of 12 heads 30.5 -> 28.5 in 32 bits, a bfloat16 prompt of
//     1,000 118 -> 109; beyond it tokens first: 25 heads in 32 bits, 600 keys (7.7 MB) 504 against 653, 8 x 1,000 keys 2,440 against
//     4,600; 12 heads of 6,000 keys (9.2 MB) 3,900 against 4,280; at 3.8 to 4.1 MB even.
// Query heads that share keys stay on one XCD: tokens first.
inline bool heads_first_pays(int n, int n_head, int n_kv_head, int hd, size_t elt, int64_t keys, int chunk, bool rows_are_requests, bool leave_splits) {
    if (n_head != n_kv_head || n > 65535) return false;
    if (rows_are_requests) return leave_splits || n > 16;
    if (chunk == 0) return true;
    int heads = n_head;
    for (int xcds = 8; xcds > 1 && heads % 2 == 0; xcds /= 2) heads /= 2;
    return heads * keys * hd * 2 * static_cast<int64_t>(elt) <= (4 << 20);
}

// (made here, so that the merges' code lies ahead of the walks' some 1.5 MB: with it behind them a batch-invariant step of 8 tokens, which merges behind each of 12
// walks, took 581.8 us, so 578.9, the instructions being the same)
template __global__ void attention_merge_kernel<float>(float* __restrict__, int64_t, const int* __restrict__, const float* __restrict__, int, int, int,
                                                       const float* __restrict__);
template __global__ void attention_merge_kernel<bf16_t>(bf16_t* __restrict__, int64_t, const int* __restrict__, const float* __restrict__, int, int, int,
                                                        const float* __restrict__);

// Whether four waves ask for the next trip's keys ahead (bfloat16). The pieces of two trips take 128 to 143 registers, three or four workgroups a
// compute unit, where one trip takes 63 to 90, five to seven: with small heads or scores to work on, whose arithmetic wants the waves, it pays until those three
// are placed (us ahead / not, 12 heads over 100 to 1,000 keys, caches not read before. Heads of 16: 64 tokens 9.9 / 10.4, 72 11.8 / 11.0, 130 18.2 / 16.9,
// 130 with a bias by distance 23.9 / 20.5; of 32: 64 tokens 15.1 / 15.9, 100 21.7 / 21.2, 130 over up to 250 keys 13.3 / 11.6. Heads of 64: 43 tokens with a sink
// 20.2 / 21.6, 64 26.8 / 26.8, 100 38.8 / 37.4, with a bias 64 32.7 / 33.5, 72 37.9 / 35.4). Heads of 64 and more with plain scores gain at any number (130 tokens
// 45.6 / 46.6).
constexpr bool next_trip_ahead_pays(bool scored, int hd, int64_t workgroups) { return (!scored && hd > 32) || workgroups <= 3 * 256; }

template <typename T, bool SCORED = false>
int launch_attention_decode(void* out, int64_t out_stride, const void* q, int64_t q_stride, const void* kc, const void* vc,
                            const int* block_tables, int max_blocks, const int* tok_list, const int* tok_seq,
                            const int* tok_pos, int n, float scale, int window, int n_head, int n_kv_head, int hd,
                            int page_size, int n_splits, int chunk, int waves, int rows_are_requests, float* partials,
                            int leave_splits, int num_pages, int reach, hipStream_t stream, float softcap = 0.0f, const float* bias_table = nullptr,
                            int max_dist = 0, const float* sinks = nullptr, int keep_first = 0) {
    int page_shift = -1, split_shift = -1;
    for (int b = 0; b < 31; ++b) {
        if ((1 << b) == page_size) page_shift = b;
        if ((1 << b) == n_splits) split_shift = b;
    }
    int64_t keys = static_cast<int64_t>(max_blocks) * page_size;
    if (reach > 0 && reach < keys) keys = reach;
    if (window > 0 && static_cast<int64_t>(window) + keep_first < keys) keys = static_cast<int64_t>(window) + keep_first;
    const int heads_first = heads_first_pays(n, n_head, n_kv_head, hd, sizeof(T), keys, chunk, rows_are_requests, leave_splits);
    const dim3 grid = heads_first ? dim3(n_head, n, n_splits) : dim3(n, n_head, n_splits);
    auto* o = static_cast<T*>(out);
    auto* pq = static_cast<const T*>(q);
    auto* pk = static_cast<const T*>(kc);
    auto* pv = static_cast<const T*>(vc);
    const bool ahead = next_trip_ahead_pays(SCORED, hd, static_cast<int64_t>(n) * n_head * n_splits);
#define LIYAB_LAUNCH(L, WAVES, U, AHEAD)                                                                                          \
    attention_decode_kernel<T, L, WAVES, U, SCORED, AHEAD><<<grid, 64 * WAVES, 0, stream>>>(                                      \
        o, out_stride, pq, q_stride, pk, pv, block_tables, max_blocks, tok_list, tok_seq, tok_pos, scale, window, n_head, n_kv_head, hd, page_size, \
        page_shift, rows_are_requests, n_splits, split_shift, chunk, partials, num_pages, heads_first, softcap, bias_table, max_dist, sinks, keep_first)
#define LIYAB_GO(L)                                                                                      \
    do {                                                                                                 \
        constexpr bool always = next_trip_ahead_pays(SCORED, 8 * L, INT64_MAX);                          \
        if (waves == 4 && ahead) LIYAB_LAUNCH(L, 4, 4, sizeof(T) == 2);                                  \
        else if (waves == 4) LIYAB_LAUNCH(L, 4, 4, sizeof(T) == 2 && always);                            \
        else if (waves == 8) LIYAB_LAUNCH(L, 8, 4, false);                                               \
        else LIYAB_LAUNCH(L, 16, sizeof(T) == 2 ? 8 : 4, false);                                         \
    } while (0)
    if (hd <= 8) LIYAB_GO(1);
    else if (hd <= 16) LIYAB_GO(2);
    else if (hd <= 32) LIYAB_GO(4);
    else if (hd <= 64) LIYAB_GO(8);
    else if (hd <= 128) LIYAB_GO(16);
    else LIYAB_GO(32);
#undef LIYAB_GO
#undef LIYAB_LAUNCH
    if (int rc = check_launch("attention_decode")) return rc;
    if (n_splits > 1 && !leave_splits) {
        attention_merge_kernel<T><<<dim3(n, n_head), ((hd + 63) / 64) * 64, 0, stream>>>(o, out_stride, tok_list, partials, n_head, hd, n_splits, sinks);
        return check_launch("attention_merge");
    }
    return 0;
}
int merge_decode_splits(bf16_t* out, int64_t out_stride, const int* tok_list, const float* partials, int n, int n_head, int hd, int n_splits, hipStream_t stream) {
    attention_merge_kernel<bf16_t><<<dim3(n, n_head), ((hd + 63) / 64) * 64, 0, stream>>>(out, out_stride, tok_list, partials, n_head, hd, n_splits);
    return check_launch("attention_merge");
}

}  // namespace liyab

using namespace liyab;

// Tokens tok_list[0..n) (or 0..n-1 when tok_list is null), each on its own. `partials` must hold
// n * n_head * n_splits * (hd + 4) floats when n_splits > 1. With `leave_splits` (n_splits > 1)
// the splits are not merged and `out` is not written: partials[token slot][head][split] holds
// hd weighted values, then the split's maximum and sum (an empty split: -inf and 0), for a
// reader that merges them as it loads them (the output projection cut over its inner dimension).
// dtype: the element type of out, q and the caches (bfloat16 or 32-bit floats). chunk: 0 = each
// split an equal share of the token's keys; > 0 = split z takes keys [z * chunk, (z + 1) * chunk)
// of the token's (n_splits * chunk must cover the longest context: keys beyond are not read).
// num_pages: the pages the caches hold; page ids of the block tables are brought into [0, num_pages).
// reach: the most keys a token of the launch has, rounded up, or 0 for what its block table holds; the order of the grid follows from
// it and nothing else does.
static int check_attention_decode(void* out, int64_t out_stride, const void* q, int64_t q_stride, const void* kc, const void* vc, int dtype,
                                  const int* block_tables, int max_blocks, const int* tok_list, const int* tok_seq, const int* tok_pos, int n,
                                  int window, int n_head, int n_kv_head, int hd, int page_size, int n_splits, int chunk, int waves,
                                  int rows_are_requests, float* partials, int leave_splits, int num_pages, int keep_first) {
    LIYAB_REQUIRE(num_pages > 0, "attention_decode: the caches hold %d pages", num_pages);
    LIYAB_REQUIRE((out || leave_splits) && q && kc && vc && block_tables && tok_seq && tok_pos, "attention_decode: null pointer");
    LIYAB_REQUIRE(dtype == kBF16 || dtype == kF32, "attention_decode: unknown dtype %d", dtype);
    LIYAB_REQUIRE(!leave_splits || n_splits > 1, "attention_decode: splits are left only when there are several");
    LIYAB_REQUIRE(n >= 0 && n_head > 0 && n_kv_head > 0 && page_size > 0 && max_blocks > 0, "attention_decode: bad sizes");
    LIYAB_REQUIRE(n_head % n_kv_head == 0, "attention_decode: %d query heads are no multiple of %d key/value heads", n_head, n_kv_head);
    LIYAB_REQUIRE(hd >= 8 && hd <= 256 && hd % 8 == 0, "attention_decode: head size %d is not a multiple of 8 in 8..256", hd);
    const int per16 = dtype == kBF16 ? 8 : 4;  // elements in 16 bytes
    LIYAB_REQUIRE(q_stride % per16 == 0 && (reinterpret_cast<uintptr_t>(q) & 15) == 0 && (reinterpret_cast<uintptr_t>(kc) & 15) == 0 &&
                      (reinterpret_cast<uintptr_t>(vc) & 15) == 0,
                  "attention_decode: queries and caches must be 16-byte aligned with a query stride that is a multiple of 16 bytes");
    LIYAB_REQUIRE(out_stride >= static_cast<int64_t>(n_head) * hd && q_stride >= static_cast<int64_t>(n_head) * hd,
                  "attention_decode: row strides are shorter than heads x head size");
    LIYAB_REQUIRE(n_splits >= 1 && n_splits <= 64 && (n_splits == 1 || partials != nullptr), "attention_decode: bad split count %d", n_splits);
    LIYAB_REQUIRE(window >= 0 && n_head <= 65535, "attention_decode: bad window or head count");
    LIYAB_REQUIRE(chunk >= 0 && keep_first >= 0, "attention_decode: a negative number of keys a split, or of kept positions");
    LIYAB_REQUIRE(chunk == 0 || n_splits > 1 || static_cast<int64_t>(chunk) * AD_LOOP_CHUNKS >= static_cast<int64_t>(max_blocks) * page_size ||
                      (window > 0 && static_cast<int64_t>(chunk) * AD_LOOP_CHUNKS >= static_cast<int64_t>(window) + keep_first),
                  "attention_decode: one workgroup walks at most %d splits of %d keys; contexts of %lld need a launch in splits", AD_LOOP_CHUNKS,
                  chunk, static_cast<long long>(max_blocks) * page_size);
    LIYAB_REQUIRE(max_blocks <= AD_MAX_BLOCKS, "attention_decode: block tables of %d pages; at most %d are taken", max_blocks, AD_MAX_BLOCKS);
    LIYAB_REQUIRE(!rows_are_requests || tok_list == nullptr, "attention_decode: rows_are_requests does not go with a row list");
    LIYAB_REQUIRE(waves == 4 || waves == 8 || waves == 16, "attention_decode: %d waves per workgroup is not 4, 8 or 16", waves);
    return 0;
}

extern "C" int liyab_attention_decode(void* out, int64_t out_stride, const void* q, int64_t q_stride, const void* kc,
                                      const void* vc, int dtype, const int* block_tables, int max_blocks, const int* tok_list,
                                      const int* tok_seq, const int* tok_pos, int n, float scale, int window,
                                      int n_head, int n_kv_head, int hd, int page_size, int n_splits, int chunk, int waves,
                                      int rows_are_requests, float* partials, int leave_splits, int num_pages, int reach, hipStream_t stream) {
    if (int rc = check_attention_decode(out, out_stride, q, q_stride, kc, vc, dtype, block_tables, max_blocks, tok_list, tok_seq, tok_pos, n, window,
                                        n_head, n_kv_head, hd, page_size, n_splits, chunk, waves, rows_are_requests, partials, leave_splits, num_pages, 0))
        return rc;
    if (n == 0) return 0;
    if (dtype == kF32)
        return launch_attention_decode<float>(out, out_stride, q, q_stride, kc, vc, block_tables, max_blocks, tok_list, tok_seq,
                                              tok_pos, n, scale, window, n_head, n_kv_head, hd, page_size, n_splits, chunk, waves,
                                              rows_are_requests, partials, leave_splits, num_pages, reach, stream);
    return launch_attention_decode<bf16_t>(out, out_stride, q, q_stride, kc, vc, block_tables, max_blocks, tok_list, tok_seq,
                                           tok_pos, n, scale, window, n_head, n_kv_head, hd, page_size, n_splits, chunk, waves,
                                           rows_are_requests, partials, leave_splits, num_pages, reach, stream);
}

// The same with the scores worked on before the softmax: softcap > 0 caps them, cap * tanh(score / cap); bias_table (float
// [max_dist + 1, n_head]) adds table[min(position - key, max_dist), head]; sinks (float [n_head], or null): exp(sinks[head])
// is added to the softmax's denominator; keep_first: positions below it stay visible behind the window.
extern "C" int liyab_attention_decode_scored(void* out, int64_t out_stride, const void* q, int64_t q_stride, const void* kc,
                                             const void* vc, int dtype, const int* block_tables, int max_blocks, const int* tok_list,
                                             const int* tok_seq, const int* tok_pos, int n, float scale, int window,
                                             int n_head, int n_kv_head, int hd, int page_size, int n_splits, int chunk, int waves,
                                             int rows_are_requests, float* partials, int leave_splits, int num_pages, int reach, float softcap,
                                             const float* bias_table, int max_dist, const float* sinks, int keep_first, hipStream_t stream) {
    if (int rc = check_attention_decode(out, out_stride, q, q_stride, kc, vc, dtype, block_tables, max_blocks, tok_list, tok_seq, tok_pos, n, window,
                                        n_head, n_kv_head, hd, page_size, n_splits, chunk, waves, rows_are_requests, partials, leave_splits, num_pages, keep_first))
        return rc;
    LIYAB_REQUIRE(softcap >= 0.0f && (bias_table == nullptr || max_dist >= 0), "attention_decode_scored: a negative cap or distance");
    LIYAB_REQUIRE(sinks == nullptr || !leave_splits, "attention_decode_scored: splits left unmerged take no sink");
    if (n == 0) return 0;
    if (dtype == kF32)
        return launch_attention_decode<float, true>(out, out_stride, q, q_stride, kc, vc, block_tables, max_blocks, tok_list, tok_seq,
                                                    tok_pos, n, scale, window, n_head, n_kv_head, hd, page_size, n_splits, chunk, waves,
                                                    rows_are_requests, partials, leave_splits, num_pages, reach, stream, softcap, bias_table, max_dist, sinks, keep_first);
    return launch_attention_decode<bf16_t, true>(out, out_stride, q, q_stride, kc, vc, block_tables, max_blocks, tok_list, tok_seq,
                                                 tok_pos, n, scale, window, n_head, n_kv_head, hd, page_size, n_splits, chunk, waves,
                                                 rows_are_requests, partials, leave_splits, num_pages, reach, stream, softcap, bias_table, max_dist, sinks, keep_first);
}

// out[m, h * hd + e] = the splits of (m, h) merged in split order: for splits that
// liyab_attention_decode left unmerged and no reader takes as they are.
extern "C" int liyab_attention_merge(void* out, int out_dtype, int64_t out_stride, const float* partials, int n, int n_head,
                                     int hd, int n_splits, hipStream_t stream) {
    LIYAB_REQUIRE(out && partials, "attention_merge: null pointer");
    LIYAB_REQUIRE(n >= 0 && n_head > 0 && n_head <= 65535 && hd > 0 && hd <= 1024 && n_splits >= 1 && n_splits <= 64, "attention_merge: bad sizes (at most 64 splits)");
    LIYAB_REQUIRE(out_stride >= static_cast<int64_t>(n_head) * hd, "attention_merge: the row stride is shorter than heads x head size");
    LIYAB_REQUIRE(out_dtype == kBF16 || out_dtype == kF32, "attention_merge: unknown dtype %d", out_dtype);
    if (n == 0) return 0;
    const dim3 grid(n, n_head);
    const int threads = ((hd + 63) / 64) * 64;
    if (out_dtype == kF32)
        attention_merge_kernel<float><<<grid, threads, 0, stream>>>(static_cast<float*>(out), out_stride, nullptr, partials, n_head, hd, n_splits);
    else
        attention_merge_kernel<bf16_t><<<grid, threads, 0, stream>>>(static_cast<bf16_t*>(out), out_stride, nullptr, partials, n_head, hd, n_splits);
    return check_launch("attention_merge");
}
