// Attention of prompt portions in 32 bits, heads of 64: the bits that attention_decode.hip leaves for each token on its own (chunk = 256 keys a split),
// from a kernel whose workgroups take 32 consecutive queries of a request to 256 of their keys.
//
// What bounds it. A token on its own is a workgroup that stages a block table, asks for its keys and absorbs them, a chain of some 8 us for
// little arithmetic, all of it on the vector unit. Here 256 keys and values lie in LDS once for 32 queries (136 KB with the queries, so a workgroup a compute unit, and eight waves, whose four parts of a row want more registers than sixteen would leave),
// and both contractions run on the matrix cores, whose v_mfma_f32_16x16x4_f32 is four fused multiply-adds one after the other. What is left is
// shared between them (1,152 cycles for 16 keys of 16 queries) and the vector unit (some 900: exponentials, maxima, the sums' trees).
// Alone, us a layer of 12 heads, token by token / here with the splits' merge: portions of 100, 237, 374 and 511 tokens 102 / 50, four of 511 183 / 77, one of 1,000
// 151 / 70, one of 500 49 / 26, eight of 33 behind 1,500 keys 133 / 84, ten of 30 17.6 / 11.3, one of 200 16.2 / 17.1, of 100 9.0 / 11.4: a workgroup is a chain of some 7 us however few
// keys it has (with a wait for each page id between the loads, a trip to memory every time, 51.7, 79, 74, 26.8, 90.6, 11.3, 17.4 and 11.8). (Eight lanes a query and the vector unit
// alone, as the other kernel, on sixteen waves: 64, 102, 94, 35, -, 15.4, 24, 15.6.)
//
// The order of a token's sums is that of the other kernel: a score is eight chains of eight dimensions, added in a tree; 32 lane groups take every 32nd
// key, four at a time, each with a maximum, a sum and weighted values of its own; groups are merged in a tree, eight to a wave, then the four waves in
// their order, then the splits. Here wave (qg, w) takes wave w's eight groups for 16 queries: a block of scores holds four groups' four keys, a group a register and a
// key a row of 16 lanes, which is how the weights enter the second contraction; the groups' parts are merged as a binary counter carries.
#include "attention_partial.h"
#include "common.h"
#include "launchers.h"

namespace liyab {

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((address_space(3))) void* lds_void_ptr;

constexpr int kRowsDim = 64, kRowsKeys = 256, kRowsQueries = 32, kRowsWaves = 8;  // head size; keys and queries a workgroup; waves: two groups of queries x four of keys

// Part of a row's keys: this lane's 16 of the weighted values, and the row's maximum and sum.
struct RowPart {
    f32x4 acc[4];
    float m, l;
};

// a <- merge(a, b), both rescaled to the larger maximum, rounded as the other kernel is compiled: merging lane groups it fuses the second part's product of the
// weighted values, merging waves the first part's (a test holds the two kernels to the same bits).
template <bool GROUPS>
__device__ __forceinline__ void merge_as_there(RowPart& a, const RowPart& b) {
#pragma clang fp contract(off)
    const float M = fmaxf(a.m, b.m);
    const float wa = a.m == -INFINITY ? 0.0f : exp_for<float>(a.m - M);
    const float wb = b.m == -INFINITY ? 0.0f : exp_for<float>(b.m - M);
    a.l = fmaf(wa, a.l, wb * b.l);
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int e = 0; e < 4; ++e) a.acc[d][e] = GROUPS ? fmaf(wb, b.acc[d][e], wa * a.acc[d][e]) : fmaf(wa, a.acc[d][e], wb * b.acc[d][e]);
    a.m = M;
}

// The values of the four rows of 16 lanes, in every row.
__device__ __forceinline__ void rows_of(float v, float (&x)[4]) {
    const auto even_odd = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);  // rows 0, 0, 2, 2 and 1, 1, 3, 3
    const auto even = __builtin_amdgcn_permlane32_swap(even_odd[0], even_odd[0], false, false);
    const auto odd = __builtin_amdgcn_permlane32_swap(even_odd[1], even_odd[1], false, false);
    x[0] = __uint_as_float(even[0]);
    x[1] = __uint_as_float(odd[0]);
    x[2] = __uint_as_float(even[1]);
    x[3] = __uint_as_float(odd[1]);
}

__global__ void __launch_bounds__(64 * kRowsWaves)
attention_rows_kernel(float* __restrict__ out, int64_t out_stride, const float* __restrict__ q, int64_t q_stride, const float* __restrict__ kc,
                      const float* __restrict__ vc, const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ work, int tile, float scale,
                      int n_head, int n_kv_head, int page_size, int page_shift, int n_splits, float* __restrict__ partials, int num_pages) {
    // keys [256][64], values [256][64], queries [32][64], in pieces of four: piece g of key k at g ^ (4 ((k / 32) % 4) + k % 4), of query i at g ^ (i % 16), so that
    // the 16 keys or queries of a block, read at one dimension, and the four keys of a group, read at 16, fall on different banks
    extern __shared__ __attribute__((aligned(1024))) float rows_lds[];
    float* const lk = rows_lds;
    float* const lv = lk + kRowsKeys * kRowsDim;
    float* const lq = lv + kRowsKeys * kRowsDim;
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int w = wave % 4, qg = wave / 4, li = lane % 16, u = lane / 16;  // this lane: query li of the wave's 16; of a group's four keys, key u
    const int h = blockIdx.x, per_tile = (tile + kRowsQueries - 1) / kRowsQueries, ti = blockIdx.y / per_tile, first_q = blockIdx.y % per_tile * kRowsQueries, z = blockIdx.z;
    const int seq = work[4 * ti], row0 = work[4 * ti + 1] + first_q, pos0 = work[4 * ti + 2] + first_q, nq = min(work[4 * ti + 3] - first_q, kRowsQueries);
    if (nq <= 0) return;
    const int mine = qg * 16 + li, row = row0 + min(mine, nq - 1);
    const bool stored = mine < nq;
    float* const part = n_splits > 1 ? partials + ((static_cast<int64_t>(row) * n_head + h) * n_splits + z) * (kRowsDim + 4) : nullptr;
    const int k_begin = z * kRowsKeys;
    const int k_hi = min(pos0 + nq - 1, static_cast<int>(min(static_cast<int64_t>(max_blocks) * page_size, static_cast<int64_t>(1) << 30)) - 1);
    if (k_begin > k_hi) {  // none of the queries sees this split's keys
        if (w == 0 && stored) {
#pragma unroll
            for (int d = 0; d < 4; ++d) *reinterpret_cast<f32x4*>(part + 16 * d + 4 * u) = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            if (u == 0) {
                part[kRowsDim] = -INFINITY;
                part[kRowsDim + 1] = 0.0f;
            }
        }
        return;
    }
    const int n_keys = min(kRowsKeys, k_hi - k_begin + 1);
    {
        // a load: four keys of 256 bytes, sixteen lanes each; the wave's loads' page ids first
        const int hkv = n_head == n_kv_head ? h : h / (n_head / n_kv_head);
        const int* const bt = block_tables + static_cast<int64_t>(seq) * max_blocks;
        constexpr int LOADS = kRowsKeys / 4 / kRowsWaves;
        int id[LOADS], off[LOADS];
#pragma unroll
        for (int l = 0; l < LOADS; ++l) {
            const int key = k_begin + min((l * kRowsWaves + wave) * 4 + u, n_keys - 1);
            const int lp = page_shift >= 0 ? key >> page_shift : key / page_size;
            off[l] = key - lp * page_size;
            id[l] = bt[lp];
        }
        const f32x4 mine_q = *reinterpret_cast<const f32x4*>(q + static_cast<int64_t>(row0 + min(tid / 16, nq - 1)) * q_stride + h * kRowsDim + li * 4);
        // (all ids are waited for here: inside the branches below, where loads into LDS are in flight that nobody can count, each would wait for everything ahead of it)
#pragma unroll
        for (int l = 0; l < LOADS; ++l) asm volatile("" : "+v"(id[l]));
#pragma unroll
        for (int l = 0; l < LOADS; ++l) {
            const int key = (l * kRowsWaves + wave) * 4;  // (a multiple of 4: its four keys differ in key % 4 = u)
            if (key >= n_keys) continue;
            // (an id outside the caches' pages becomes one that exists: whatever a table holds, no fetch leaves the caches)
            const int piece = li ^ (4 * ((key >> 5) & 3) + u);
            const int64_t at = ((static_cast<int64_t>(min(max(id[l], 0), num_pages - 1)) * n_kv_head + hkv) * page_size + off[l]) * kRowsDim + piece * 4;
            const float *from_k = kc + at, *from_v = vc + at;
            float *to_k = lk + key * kRowsDim, *to_v = lv + key * kRowsDim;
            __builtin_amdgcn_global_load_lds(from_k, (lds_void_ptr)(to_k), 16, 0, 0);
            __builtin_amdgcn_global_load_lds(from_v, (lds_void_ptr)(to_v), 16, 0, 0);
        }
        *reinterpret_cast<f32x4*>(lq + tid / 16 * kRowsDim + (li ^ (tid / 16 & 15)) * 4) = mine_q;
    }
    __syncthreads();

    // keys of the split that this lane's query sees, and the fewest and the most among the wave's
    const int seen = min(pos0 + min(mine, nq - 1) + 1 - k_begin, n_keys);
    const int least = min(pos0 + min(qg * 16, nq - 1) + 1 - k_begin, n_keys), most = qg * 16 < nq ? min(pos0 + min(qg * 16 + 15, nq - 1) + 1 - k_begin, n_keys) : 0;
    RowPart sum, one, two;  // all groups merged so far by fours; the last group, the last pair, waiting for their partners
    sum.m = -INFINITY;
    sum.l = 0.0f;
#pragma unroll
    for (int d = 0; d < 4; ++d) sum.acc[d] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
    for (int x = 0; x < 2; ++x) {
        // groups 4 x .. 4 x + 3 of wave w, keys first .. first + 3, and every 32nd from there on
        const int first = w * 8 + 4 * x;
        if (first >= most) break;  // (no query of the wave sees a key of them: merged, they would change nothing)
        const int trips = first + 128 < most ? 2 : 1;
        f32x4 s[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            if (t >= trips) break;
            const int j = first + 128 * t;
            const float* const key = lk + (j + 32 * (li >> 2) + (li & 3)) * kRowsDim + u;
            const float* const query = lq + mine * kRowsDim + u;
            f32x4 tree[3];
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int g = 2 * c; g < 2 * c + 2; ++g) v = __builtin_amdgcn_mfma_f32_16x16x4f32(key[(g ^ li) * 4], query[(g ^ li) * 4], v, 0, 0, 0);
                if ((c & 1) == 0) tree[0] = v;
                else {
                    v = tree[0] + v;
                    if ((c & 2) == 0) tree[1] = v;
                    else {
                        v = tree[1] + v;
                        if ((c & 4) == 0) tree[2] = v;
                        else s[t] = tree[2] + v;
                    }
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                s[t][r] = s[t][r] * scale;
                s[t][r] = j + 32 * u + r < seen ? s[t][r] : -INFINITY;
            }
        }
        const bool whole = first + 3 + 96 + 128 * (trips - 1) < least;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
#pragma clang fp contract(off)
            RowPart st;
            st.m = -INFINITY;
            st.l = 0.0f;
#pragma unroll
            for (int d = 0; d < 4; ++d) st.acc[d] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                if (t >= trips) break;
                float v[4];
                rows_of(s[t][r], v);
                const float m_new = fmaxf(fmaxf(fmaxf(fmaxf(st.m, v[0]), v[1]), v[2]), v[3]);
                const float ref = m_new == -INFINITY ? 0.0f : m_new;
                if (t > 0) {  // (the first time there is nothing to rescale)
                    const float corr = exp_for<float>(st.m - ref);
                    st.l *= corr;
#pragma unroll
                    for (int d = 0; d < 4; ++d) st.acc[d] *= corr;
                }
                const float p = exp_for<float>(s[t][r] - ref);
                rows_of(p, v);
#pragma unroll
                for (int k = 0; k < 4; ++k) st.l += v[k];
                const int at = first + 128 * t + 32 * u + r;
                const float* const value = lv + at * kRowsDim + (li & 3);
                float vf[4];
#pragma unroll
                for (int d = 0; d < 4; ++d) vf[d] = value[((4 * d + (li >> 2)) ^ (4 * u + r)) * 4];
                bool odd = false;  // a value that is no number where not every query sees its key: 0 times it would be none either
                if (!whole) {
#pragma unroll
                    for (int d = 0; d < 4; ++d) {
                        vf[d] = at < n_keys ? vf[d] : 0.0f;
                        odd = odd || !(fabsf(vf[d]) < INFINITY);
                    }
                }
                if (__builtin_amdgcn_ballot_w64(odd) == 0) {
#pragma unroll
                    for (int d = 0; d < 4; ++d) st.acc[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[d], p, st.acc[d], 0, 0, 0);
                } else {
                    // such values come last, to those who see them: what they leave is no number, or infinite, in any order
#pragma unroll
                    for (int d = 0; d < 4; ++d) st.acc[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(fabsf(vf[d]) < INFINITY ? vf[d] : 0.0f, p, st.acc[d], 0, 0, 0);
                    for (int k = 0; k < 4; ++k) {
                        const int its = first + 128 * t + 32 * k + r;
                        if (its >= seen) continue;
#pragma unroll
                        for (int d = 0; d < 4; ++d)
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                const float x_value = lv[its * kRowsDim + (((4 * d + u) ^ (4 * k + r)) * 4) + e];
                                const float x_p = k == 0 ? v[0] : k == 1 ? v[1] : k == 2 ? v[2] : v[3];
                                if (!(fabsf(x_value) < INFINITY)) st.acc[d][e] += x_p * x_value;
                            }
                    }
                }
                st.m = m_new;
            }
            if (r == 0) one = st;
            else if (r == 1) {
                merge_as_there<true>(one, st);
                two = one;
            } else if (r == 2) one = st;
            else {
                merge_as_there<true>(one, st);
                merge_as_there<true>(two, one);
            }
        }
        if (x == 0) sum = two;
        else merge_as_there<true>(sum, two);
    }
    __syncthreads();  // (the sums take the keys' place)
    float* const red = rows_lds + wave * 18 * 64 + lane;
    if (w > 0) {
        red[0] = sum.m;
        red[64] = sum.l;
#pragma unroll
        for (int e = 0; e < 16; ++e) red[(2 + e) * 64] = sum.acc[e / 4][e % 4];
    }
    __syncthreads();
    if (w != 0 || !stored) return;
#pragma unroll 1
    for (int other = 1; other < 4; ++other) {
        RowPart b;
        b.m = red[other * 18 * 64];
        b.l = red[other * 18 * 64 + 64];
#pragma unroll
        for (int e = 0; e < 16; ++e) b.acc[e / 4][e % 4] = red[other * 18 * 64 + (2 + e) * 64];
        merge_as_there<false>(sum, b);
    }
    if (n_splits == 1) {
        float* const o = out + static_cast<int64_t>(row) * out_stride + h * kRowsDim + 4 * u;
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
            for (int e = 0; e < 4; ++e) o[16 * d + e] = sum.acc[d][e] / sum.l;
    } else {
#pragma unroll
        for (int d = 0; d < 4; ++d) *reinterpret_cast<f32x4*>(part + 16 * d + 4 * u) = sum.acc[d];
        if (u == 0) {
            part[kRowsDim] = sum.m;
            part[kRowsDim + 1] = sum.l;
        }
    }
}

}  // namespace liyab

using namespace liyab;

// Tiles work[n_tiles][4] = (request, first row, first position, queries: up to `tile`, 32, 64 or 128) of 32-bit queries over 32-bit caches of heads of 64, each token over its keys
// 0 .. position. n_splits: splits of 256 keys, as many as the longest context has; with one, rows of `out` are written; with more, partials[row][head][split][68]: 64
// weighted values, the split's maximum and sum (an empty split: -inf and 0), for liyab_attention_merge. The caller has checked the tiles' rows against q, out and partials.
extern "C" int liyab_attention_rows(float* out, int64_t out_stride, const float* q, int64_t q_stride, const float* kc, const float* vc, const int* block_tables,
                                    int max_blocks, const int* work, int n_tiles, int tile, float scale, int n_head, int n_kv_head, int page_size, int n_splits,
                                    float* partials, int num_pages, hipStream_t stream) {
    LIYAB_REQUIRE(q && kc && vc && block_tables && work && (n_splits > 1 ? partials != nullptr : out != nullptr), "attention_rows: null pointer");
    LIYAB_REQUIRE(num_pages > 0 && n_tiles >= 0 && n_head > 0 && n_head <= 65535 && n_kv_head > 0 && n_head % n_kv_head == 0 && page_size > 0 && max_blocks > 0,
                  "attention_rows: bad sizes");
    LIYAB_REQUIRE(tile == 32 || tile == 64 || tile == 128, "attention_rows: tiles of %d queries are not 32, 64 or 128", tile);
    LIYAB_REQUIRE(n_splits >= 1 && n_splits <= 64 && static_cast<int64_t>(n_tiles) * (tile / kRowsQueries) <= 65535, "attention_rows: %d splits, %d tiles", n_splits, n_tiles);
    LIYAB_REQUIRE(q_stride % 4 == 0 && (reinterpret_cast<uintptr_t>(q) & 15) == 0 && (reinterpret_cast<uintptr_t>(kc) & 15) == 0 && (reinterpret_cast<uintptr_t>(vc) & 15) == 0,
                  "attention_rows: queries and caches must be 16-byte aligned with a query stride that is a multiple of 4");
    LIYAB_REQUIRE((reinterpret_cast<uintptr_t>(partials) & 15) == 0, "attention_rows: partials must be 16-byte aligned");
    LIYAB_REQUIRE(q_stride >= static_cast<int64_t>(n_head) * kRowsDim && (n_splits > 1 || out_stride >= static_cast<int64_t>(n_head) * kRowsDim), "attention_rows: short rows");
    if (n_tiles == 0) return 0;
    constexpr int smem = (2 * kRowsKeys + kRowsQueries) * kRowsDim * 4;
    static bool ready = false;  // once, outside any stream capture's first use
    if (!ready) {
        hipFuncSetAttribute(reinterpret_cast<const void*>(attention_rows_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, smem);
        ready = true;
    }
    int page_shift = -1;
    for (int b = 0; b < 31; ++b)
        if ((1 << b) == page_size) page_shift = b;
    attention_rows_kernel<<<dim3(n_head, n_tiles * (tile / kRowsQueries), n_splits), 64 * kRowsWaves, smem, stream>>>(
        out, out_stride, q, q_stride, kc, vc, block_tables, max_blocks, work, tile, scale, n_head, n_kv_head, page_size, page_shift, n_splits, partials, num_pages);
    return check_launch("attention_rows");
}
