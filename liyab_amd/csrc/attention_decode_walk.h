// Attention of one token's head over paged keys and values, a split of them (attention_decode.hip says how and why): what its kernel and the one that takes
// prompt portions beside such tokens (attention_mixed.hip) share.
#pragma once
#include <type_traits>

#include "attention_partial.h"
#include "common.h"

namespace liyab {

typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

constexpr int AD_MAX_BLOCKS = 2048;  // page ids of a request kept in LDS
constexpr int AD_LOOP_CHUNKS = 16;   // splits by position that one workgroup walks in turn, at most


__device__ __forceinline__ void unpack8(const u32x4& v, float* f) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        f[2 * i] = __uint_as_float(v[i] << 16);
        f[2 * i + 1] = __uint_as_float(v[i] & 0xffff0000u);
    }
}

// 8 consecutive elements of a row as they are loaded (bfloat16 stays packed until it is used), and as floats
typedef __attribute__((ext_vector_type(4))) float f32x4;
struct Raw8F { f32x4 a, b; };
__device__ __forceinline__ u32x4 fetch8(const bf16_t* p) { return *reinterpret_cast<const u32x4*>(p); }
__device__ __forceinline__ Raw8F fetch8(const float* p) {
    return Raw8F{*reinterpret_cast<const f32x4*>(p), *reinterpret_cast<const f32x4*>(p + 4)};
}
__device__ __forceinline__ void unpack8(const Raw8F& v, float* f) {
#pragma unroll
    for (int i = 0; i < 4; ++i) { f[i] = v.a[i]; f[4 + i] = v.b[i]; }
}
template <typename T> struct Raw8 { typedef u32x4 type; };
template <> struct Raw8<float> { typedef Raw8F type; };
// A sink joins a row's softmax: a learned logit a head that stands in the denominator once, as a key would whose score it is,
// and has no value. (m, l, acc): the row's maximum, sum and weighted values, rescaled to the larger of m and the sink.
template <typename T, int N = 8>
__device__ __forceinline__ void add_sink(float& m, float& l, float (&acc)[N], float sink) {
    const float M = fmaxf(m, sink);
    const float w = m == -INFINITY ? 0.0f : exp_for<T>(m - M);
    l = l * w + exp_for<T>(sink - M);
#pragma unroll
    for (int e = 0; e < N; ++e) acc[e] *= w;
    m = M;
}

// Splits of rows tok_list[0..n) in bfloat16, merged in their order (attention_decode.hip).
int merge_decode_splits(bf16_t* out, int64_t out_stride, const int* tok_list, const float* partials, int n, int n_head, int hd, int n_splits, hipStream_t stream);

// (aligned as arrays on their own would be: a part's ten floats are read in pieces of eight bytes)
template <int LPK, int AD_WAVES>
struct alignas(16) DecodeLds {
    alignas(16) float sums[2][AD_WAVES][LPK][10];  // the waves' sums, for the first wave to merge; two of them in turn, so that one barrier a split is enough
    alignas(16) int pages[AD_MAX_BLOCKS];
    alignas(16) float stash[AD_LOOP_CHUNKS][LPK][10];
};

// SCORED: the score scale * q . k is worked on before the softmax: a soft cap, cap * tanh(score / cap) (softcap > 0), then
// a bias by distance, bias_table[min(position - key, max_dist), head] (bias_table given); `sinks` (one logit a head) join the
// softmax's denominator where the row's sums are final; with a window, the first `keep_first` positions may stay visible: the
// walk goes over places first - kept .. position, of which those ahead of `first` are positions 0 .. kept - 1. Without SCORED these arguments are not read.
// AHEAD: the next trip's keys are on their way while this one's are absorbed (where it pays: next_trip_ahead_pays).
template <typename T, int LPK, int AD_WAVES, int AD_U, bool SCORED, bool AHEAD>
__device__ __forceinline__ void attention_decode_walk(DecodeLds<LPK, AD_WAVES>& shared, int slot, int h, int z,
                        T* __restrict__ out, int64_t out_stride, const T* __restrict__ q, int64_t q_stride,
                        const T* __restrict__ kc, const T* __restrict__ vc,
                        const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ tok_list,
                        const int* __restrict__ tok_seq, const int* __restrict__ tok_pos, float scale, int window,
                        int n_head, int n_kv_head, int hd, int page_size, int page_shift, int rows_are_requests,
                        int n_splits, int split_shift, int chunk, float* __restrict__ partials, int num_pages, float softcap,
                        const float* __restrict__ bias_table, int max_dist, const float* __restrict__ sinks, int keep_first) {
    constexpr int KPP = 64 / LPK;  // keys per wave and pass
    constexpr int TRIP = AD_WAVES * KPP * AD_U;
    constexpr bool BY_PASS = SCORED || LPK <= 4;  // a wave leaves out the passes behind its last key too: where one is much arithmetic, or many keys
    typedef typename Raw8<T>::type Raw;
    typedef std::integral_constant<bool, true> Whole;  // every lane has keys throughout the trip
    typedef std::integral_constant<bool, false> Ragged;
    auto& sbt = shared.pages;
    auto& stash = shared.stash;
    const int t = tok_list != nullptr ? tok_list[slot] : slot;
    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    const int c = lane % LPK, kg = lane / LPK;
    const bool active = c * 8 < hd;
    // The request's page ids go to LDS first, so that fetching a key is one load deep; they are
    // loaded together with the position and the query (when every row is its own request the
    // block-table row is known without looking the request up).
    const int seq = rows_are_requests ? t : tok_seq[t];
    const int* bt = block_tables + static_cast<int64_t>(seq) * max_blocks;
    // (an id outside the caches' pages, an unmapped -1 or a wrong word, becomes a page that exists:
    // whatever a table holds, no fetch leaves the caches)
    for (int i = tid; i < max_blocks; i += 64 * AD_WAVES) sbt[i] = min(max(bt[i], 0), num_pages - 1);
    // (a position past the block table's reach would index the staged ids out of range)
    const int pos = static_cast<int>(min(static_cast<int64_t>(max(tok_pos[t], 0)), static_cast<int64_t>(max_blocks) * page_size - 1));
    const int hkv = n_head == n_kv_head ? h : h / (n_head / n_kv_head);
    const int64_t page_stride = static_cast<int64_t>(n_kv_head) * page_size * hd;
    // lanes past the head dimension read column 0 and multiply it by a zero query
    const int col = active ? c * 8 : 0;
    float qf[8];
    unpack8(fetch8(q + static_cast<int64_t>(t) * q_stride + static_cast<int64_t>(h) * hd + col), qf);
    if (!active) {
#pragma unroll
        for (int e = 0; e < 8; ++e) qf[e] = 0.0f;
    }
    const int64_t head_off = static_cast<int64_t>(hkv) * page_size * hd + col;
    __syncthreads();
    const int first_seen = window > 0 ? max(0, pos - window + 1) : 0;  // the window's first position
    const int first = SCORED ? first_seen - min(keep_first, first_seen) : first_seen;  // the walk's first place
    const int n_keys = pos - first + 1;
    // Splits by position launched as one (chunk > 0, n_splits == 1): the workgroup walks the token's
    // splits one after the other, keeps each one's sums apart and merges them at the end as the merge
    // kernel would, operation for operation: the bits of the split launch without its traffic, for
    // steps of many tokens.
    const bool walks_all = chunk > 0 && n_splits == 1;
    const int z_count = walks_all ? min(AD_LOOP_CHUNKS, max(1, (n_keys + chunk - 1) / chunk)) : 1;  // (the launcher has checked that they fit)
    for (int zi = 0; zi < z_count; ++zi) {
    float (&lds)[AD_WAVES][LPK][10] = shared.sums[zi & 1];
    const int zz = walks_all ? zi : z;
    // split zz: its share of the keys, or keys [zz * chunk, (zz + 1) * chunk) of them (none, for a short context)
    const auto share = [&](int z0) {  // the keys ahead of split z0: a shift where the splits are a power of two (a 64-bit division is a hundred instructions)
        const int64_t all = static_cast<int64_t>(n_keys) * z0;
        return static_cast<int>(split_shift >= 0 ? all >> split_shift : all / n_splits);
    };
    const int k_begin = first + (chunk > 0 ? zz * chunk : share(zz));
    const int k_end = chunk > 0 ? min(pos + 1, k_begin + chunk) : first + share(zz + 1);
    Partial st;
    st.m = -INFINITY;
    st.l = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) st.acc[e] = 0.0f;

    // The walk, TRIP keys of the workgroup a trip: lane group kg of wave w takes keys j0 + (u AD_WAVES + w) KPP + kg.
    const auto fetch = [&](int j0, Raw (&kv)[AD_U], Raw (&vv)[AD_U]) {
#pragma unroll
        for (int u = 0; u < AD_U; ++u) {
            // (past the split a mapped position, whose values are not used; no branch around the loads: a load under a branch is
            // waited for where the branch ends)
            int jc = j0 + (u * AD_WAVES + wave) * KPP + kg;
            jc = jc < k_end ? jc : pos;
            if constexpr (SCORED) jc = jc < first_seen ? jc - first : jc;
            const int lp = page_shift >= 0 ? jc >> page_shift : jc / page_size;
            const int off = page_shift >= 0 ? jc & (page_size - 1) : jc - lp * page_size;
            const int64_t at = static_cast<int64_t>(sbt[lp]) * page_stride + head_off + static_cast<int64_t>(off) * hd;
            kv[u] = fetch8(kc + at);
            vv[u] = fetch8(vc + at);
        }
    };
    // A wave's walk ends with its own last key: a trip is up to 4,096 keys, of which short contexts and windows fill little
    // (32 tokens of 12 heads of 64 in a window of 256 with 4 kept, 8 waves: 11.5 us with every wave in every trip, 10.0 so).
    const int own = __builtin_amdgcn_readfirstlane(wave) * KPP;
    const auto has = [&](int j0, int u) { return j0 + u * AD_WAVES * KPP + own < k_end; };  // pass u of the trip from j0 on has a key of this wave
    const auto absorb = [&](auto whole, int j0, const Raw (&kv)[AD_U], Raw (&vv)[AD_U]) {
#pragma clang fp contract(off)  // a whole trip and a ragged one round alike: nothing is fused but what says so
        float s[AD_U];
        float m_new = st.m;
#pragma unroll
        for (int u = 0; u < AD_U; ++u) {
            if (BY_PASS && !decltype(whole)::value && !has(j0, u)) break;
            float kf[8];
            unpack8(kv[u], kf);
            float d = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; ++e) d = fmaf(kf[e], qf[e], d);
            s[u] = group_sum<LPK>(d) * scale;  // over the lanes that share the key
            const int place = j0 + (u * AD_WAVES + wave) * KPP + kg;
            if constexpr (SCORED) {
                if (softcap > 0.0f) s[u] = softcap * tanhf(s[u] / softcap);
                if (bias_table != nullptr) s[u] += bias_table[static_cast<int64_t>(max(0, min(pos - (place < first_seen ? place - first : place), max_dist))) * n_head + h];
            }
            if constexpr (!decltype(whole)::value) {
                if (place >= k_end) {
                    s[u] = -INFINITY;
                    vv[u] = Raw{};  // (its weight is 0, and 0 times an infinity would be no number)
                }
            }
            m_new = fmaxf(m_new, s[u]);
        }
        // (a lane group without a key so far: every exponential below is 0)
        const float ref = m_new == -INFINITY ? 0.0f : m_new;
        const float corr = exp_for<T>(st.m - ref);
        st.l *= corr;
#pragma unroll
        for (int e = 0; e < 8; ++e) st.acc[e] *= corr;
#pragma unroll
        for (int u = 0; u < AD_U; ++u) {
            if (BY_PASS && !decltype(whole)::value && !has(j0, u)) break;
            const float p = exp_for<T>(s[u] - ref);
            st.l += p;
            float vf[8];
            unpack8(vv[u], vf);
#pragma unroll
            for (int e = 0; e < 8; ++e) st.acc[e] = fmaf(p, vf[e], st.acc[e]);
        }
        st.m = m_new;
    };
    if (has(k_begin, 0)) {
        Raw ka[AD_U], va[AD_U];
        int j0 = k_begin;
        if constexpr (AHEAD) {
            Raw kb[AD_U], vb[AD_U];
            fetch(j0, ka, va);
            // (fences for the scheduler, which would sink the loads to their use)
            for (;;) {
                if (!has(j0 + TRIP, 0)) {
                    absorb(Ragged{}, j0, ka, va);
                    break;
                }
                fetch(j0 + TRIP, kb, vb);
                __builtin_amdgcn_sched_barrier(0);
                absorb(Whole{}, j0, ka, va);
                __builtin_amdgcn_sched_barrier(0);
                j0 += TRIP;
                if (!has(j0 + TRIP, 0)) {
                    absorb(Ragged{}, j0, kb, vb);
                    break;
                }
                fetch(j0 + TRIP, ka, va);
                __builtin_amdgcn_sched_barrier(0);
                absorb(Whole{}, j0, kb, vb);
                __builtin_amdgcn_sched_barrier(0);
                j0 += TRIP;
            }
        } else {
            for (; has(j0 + TRIP, 0); j0 += TRIP) {
                fetch(j0, ka, va);
                absorb(Whole{}, j0, ka, va);
            }
            fetch(j0, ka, va);
            absorb(Ragged{}, j0, ka, va);
        }
    }
    // lane groups of the wave, in a fixed tree
#pragma unroll
    for (int off = LPK; off < 64; off <<= 1) {
        const float mo = __shfl_xor(st.m, off, 64), lo = __shfl_xor(st.l, off, 64);
        float ao[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) ao[e] = __shfl_xor(st.acc[e], off, 64);
        merge_partial<T, AD_U == 8>(st, mo, lo, ao);
    }
    if (kg == 0) {
        lds[wave][c][0] = st.m;
        lds[wave][c][1] = st.l;
#pragma unroll
        for (int e = 0; e < 8; ++e) lds[wave][c][2 + e] = st.acc[e];
    }
    __syncthreads();
    if (wave == 0 && kg == 0 && active) {
#pragma unroll
        for (int w = 1; w < AD_WAVES; ++w) merge_partial<T, true>(st, lds[w][c][0], lds[w][c][1], &lds[w][c][2]);
        if (z_count > 1) {
            stash[zi][c][0] = st.m;
            stash[zi][c][1] = st.l;
#pragma unroll
            for (int e = 0; e < 8; ++e) stash[zi][c][2 + e] = st.acc[e];
        } else if (n_splits == 1) {
            T* o = out + static_cast<int64_t>(t) * out_stride + static_cast<int64_t>(h) * hd + c * 8;
            if constexpr (SCORED) {
                if (sinks != nullptr) add_sink<T>(st.m, st.l, st.acc, sinks[h]);
            }
            if (chunk > 0) {
                // as the merge of several splits divides: a token has the same bits alone in one split
                // and beside longer contexts, its later splits empty
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e] = from_float<T>(st.acc[e] / st.l);
            } else {
                const float inv = 1.0f / st.l;
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e] = from_float<T>(st.acc[e] * inv);
            }
        } else {
            // partials [token slot][head][split][hd + 4]: values, then maximum and sum (and two
            // unused, which keep every split's values 16-byte aligned)
            float* p = partials + ((static_cast<int64_t>(slot) * n_head + h) * n_splits + z) * (hd + 4);
#pragma unroll
            for (int e = 0; e < 8; ++e) p[c * 8 + e] = st.acc[e];
            if (c == 0) {
                p[hd] = st.m;
                p[hd + 1] = st.l;
            }
        }
    }
    }
    if (z_count > 1 && wave == 0 && kg == 0 && active) {
        // (each lane reads what it wrote itself)
        float M = -INFINITY;
        for (int zi = 0; zi < z_count; ++zi) M = fmaxf(M, stash[zi][c][0]);
        float sum = 0.0f, o[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = 0.0f;
        for (int zi = 0; zi < z_count; ++zi) {
            const float m = stash[zi][c][0];
            if (m == -INFINITY) continue;
            const float w = exp_for<T>(m - M);
            sum = fmaf(w, stash[zi][c][1], sum);
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = fmaf(w, stash[zi][c][2 + e], o[e]);
        }
        if constexpr (SCORED) {
            if (sinks != nullptr) add_sink<T>(M, sum, o, sinks[h]);
        }
        T* dst = out + static_cast<int64_t>(t) * out_stride + static_cast<int64_t>(h) * hd + c * 8;
#pragma unroll
        for (int e = 0; e < 8; ++e) dst[e] = from_float<T>(o[e] / sum);
    }
}

}  // namespace liyab
