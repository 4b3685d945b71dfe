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
#include <type_traits>

#include "attention_partial.h"
#include "common.h"
#include "launchers.h"

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

// SCORED: the score scale * q . k is worked on before the softmax: a soft cap, cap * tanh(score / cap) (softcap > 0), then
// a bias by distance, bias_table[min(position - key, max_dist), head] (bias_table given); `sinks` (one logit a head) join the
// softmax's denominator where the row's sums are final; with a window, the first `keep_first` positions may stay visible: the
// walk goes over places first - kept .. position, of which those ahead of `first` are positions 0 .. kept - 1. Without SCORED these arguments are not read, and the kernel is the one it was.
// AHEAD: the next trip's keys are on their way while this one's are absorbed (where it pays: next_trip_ahead_pays).
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
    constexpr int KPP = 64 / LPK;  // keys per wave and pass
    constexpr int TRIP = AD_WAVES * KPP * AD_U;
    constexpr bool BY_PASS = SCORED || LPK <= 4;  // a wave leaves out the passes behind its last key too: where one is much arithmetic, or many keys
    typedef typename Raw8<T>::type Raw;
    typedef std::integral_constant<bool, true> Whole;  // every lane has keys throughout the trip
    typedef std::integral_constant<bool, false> Ragged;
    __shared__ float lds2[2][AD_WAVES][LPK][10];  // the waves' sums, for the first wave to merge; two of them in turn, so that one barrier a split is enough
    // (which of the two the grid runs along first: heads_first_pays)
    const int slot = heads_first ? blockIdx.y : blockIdx.x;
    const int t = tok_list != nullptr ? tok_list[slot] : slot;
    const int h = heads_first ? blockIdx.x : blockIdx.y, z = blockIdx.z;
    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    const int c = lane % LPK, kg = lane / LPK;
    const bool active = c * 8 < hd;
    // The request's page ids go to LDS first, so that fetching a key is one load deep; they are
    // loaded together with the position and the query (when every row is its own request the
    // block-table row is known without looking the request up).
    __shared__ int sbt[AD_MAX_BLOCKS];
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
    __shared__ float stash[AD_LOOP_CHUNKS][LPK][10];
    for (int zi = 0; zi < z_count; ++zi) {
    float (&lds)[AD_WAVES][LPK][10] = lds2[zi & 1];
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
        merge_partial<T>(st, mo, lo, ao);
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
        for (int w = 1; w < AD_WAVES; ++w) merge_partial<T>(st, lds[w][c][0], lds[w][c][1], &lds[w][c][2]);
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
