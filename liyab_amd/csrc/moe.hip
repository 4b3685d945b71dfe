// Routing of a mixture of experts: who goes where, before the experts' products run
// (grouped_product.hip).
//
// liyab_moe_route: from each token's 32-bit router logits the `top` experts with the largest
// logits (among equal logits the lower number first) and their weights, the softmax over the chosen
// logits alone, in 32-bit. ids and weights [n, top]: entry t * top + k is token t's k-th choice.
// mode 1: the choice among groups of experts instead (route_token_groups): softmax over all experts, the best
// groups only, weights divided by their sum.
// mode 2: scores s = 1 / (1 + exp(-z)), the choice by c = s + correction (route_wave): a group's score is the sum of its two
// largest c, only experts of the best groups, of those the `top` largest c; weights are the chosen s as they are. A wave routes a
// token (its scores in LDS, an expert a lane), since every score costs an exponential.
// mode 3: as mode 2 with scores s = softmax(z) over all outputs; weights are scale * s of the chosen ones.
// Modes 2 and 3: outputs from `n_listed` on are identity experts, whose result is the token's own input: they get the id -1, so that no
// list holds them, and whoever adds a token's rows up puts the input there. With `extra`, a token has one more entry behind its `top`: expert
// n_listed, which every token takes, weighted sigmoid(z[E]) (a logit of its own behind the router's).
//
// liyab_moe_align: the entries listed by expert, each expert's stretch padded to whole tiles of
// `block` places: rows_list [max_tiles * block] (an entry's number, -1 for an empty place) and
// tile_group [max_tiles] (the expert of each tile, -1 for a tile that is not used). max_tiles is
// a bound that the step's sizes fix (entries / block + min(experts, entries), rounded up), so
// that the products' grids do not depend on where the tokens went. One workgroup.
//
// liyab_moe_route_align: both in one launch, for steps of at most 1,024 tokens (modes 2 and 3: kWaveRouteTokens).
#include "common.h"
#include "launchers.h"

namespace liyab {

constexpr int kMaxTop = 64;

// One token's choice: the `top` largest of its E logits (the lower number among equals) and the softmax over them.
__device__ __forceinline__ void route_token(const float* __restrict__ z, int E, int top, int* __restrict__ ids, float* __restrict__ weights) {
    int chosen[kMaxTop];
    float value[kMaxTop];
    for (int k = 0; k < top; ++k) {
        int best = -1;
        float bv = 0.0f;
        for (int e = 0; e < E; ++e) {
            bool taken = false;
            for (int j = 0; j < k; ++j) taken = taken || chosen[j] == e;
            const float v = z[e];
            if (!taken && (best < 0 || v > bv)) {
                best = e;
                bv = v;
            }
        }
        chosen[k] = best;
        value[k] = bv;
    }
    float sum = 0.0f;
    const float largest = value[0];  // the first choice holds the largest logit
    for (int k = 0; k < top; ++k) {
        value[k] = expf(value[k] - largest);
        sum += value[k];
    }
    for (int k = 0; k < top; ++k) {
        ids[k] = chosen[k];
        weights[k] = value[k] / sum;
    }
}

// One token's choice among groups of experts: s = softmax(z) over all experts; the experts form `n_groups` equal groups of
// neighbours, a group's score is its largest s, and only experts of the `keep` best groups (the lower number among equals)
// can be chosen; of those the `top` largest s (the lower number among equals), weighted s / (their sum + 1e-20).
constexpr int kMaxGroups = 64;
constexpr float kWeightFloor = 1e-20f;

__device__ __forceinline__ void route_token_groups(const float* __restrict__ z, int E, int top, int n_groups, int keep, int* __restrict__ ids,
                                                   float* __restrict__ weights) {
    float largest = z[0];
    for (int e = 1; e < E; ++e) largest = fmaxf(largest, z[e]);
    float total = 0.0f;
    for (int e = 0; e < E; ++e) total += expf(z[e] - largest);
    const int per = E / n_groups;
    uint64_t kept = 0;  // the groups whose experts can be chosen
    for (int k = 0; k < keep; ++k) {
        int best = -1;
        float bv = 0.0f;
        for (int g = 0; g < n_groups; ++g) {
            if ((kept >> g) & 1) continue;
            float gv = z[g * per];
            for (int e = 1; e < per; ++e) gv = fmaxf(gv, z[g * per + e]);  // (the largest score is the largest logit's)
            if (best < 0 || gv > bv) {
                best = g;
                bv = gv;
            }
        }
        kept |= uint64_t(1) << best;
    }
    int chosen[kMaxTop];
    float value[kMaxTop];
    float sum = 0.0f;
    for (int k = 0; k < top; ++k) {
        int best = -1;
        float bv = 0.0f;
        for (int e = 0; e < E; ++e) {
            if (!((kept >> (e / per)) & 1)) continue;
            bool taken = false;
            for (int j = 0; j < k; ++j) taken = taken || chosen[j] == e;
            const float v = z[e];
            if (!taken && (best < 0 || v > bv)) {
                best = e;
                bv = v;
            }
        }
        chosen[k] = best;
        value[k] = expf(bv - largest) / total;
        sum += value[k];
    }
    for (int k = 0; k < top; ++k) {
        ids[k] = chosen[k];
        weights[k] = value[k] / (sum + kWeightFloor);
    }
}

// One token's choice by a wave, c (LDS, E floats) its own: see mode 2 above. Among equals the lower number first; an expert that
// cannot be chosen, or has been, is minus infinity (c itself can be negative).
constexpr int kMaxWaveExperts = 2048;
constexpr int kWaveRouteTokens = 64;  // tokens a launch of one workgroup routes at most (sixteen waves, four each)

// What a wave's lanes wrote to LDS is there for its other lanes.
__device__ __forceinline__ void wave_lds_order() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

struct RouteArgs {
    int mode, n_groups, keep;
    const float* correction;
    float scale;          // mode 3: on the weights
    int n_listed, extra;  // modes 2 and 3: see the head of this file
};

__device__ __forceinline__ void route_wave(const float* __restrict__ z, const RouteArgs& ra, int E, int top, int* __restrict__ ids, float* __restrict__ weights,
                                           float* c) {
    const int lane = threadIdx.x % kWave, n_groups = ra.n_groups, keep = ra.keep;
    const float* correction = ra.correction;
    float largest = 0.0f, norm = 1.0f;  // mode 3: a score is exp(z - largest) * norm
    if (ra.mode == 3) {
        largest = -INFINITY;
        for (int e = lane; e < E; e += kWave) largest = fmaxf(largest, z[e]);
        largest = wave_max(largest);
        float total = 0.0f;
        for (int e = lane; e < E; e += kWave) total += expf(z[e] - largest);
        norm = 1.0f / wave_sum(total);
    }
    auto score = [&](int e) { return ra.mode == 3 ? expf(z[e] - largest) * norm : 1.0f / (1.0f + expf(-z[e])); };
    for (int e = lane; e < E; e += kWave) c[e] = score(e) + (correction != nullptr ? correction[e] : 0.0f);
    wave_lds_order();
    const int per = E / n_groups;
    uint64_t kept = ~uint64_t(0);
    if (keep < n_groups) {
        kept = 0;
        float score = -INFINITY;  // lane g: group g's
        if (lane < n_groups) {
            float a = -INFINITY, b = -INFINITY;  // its two largest
            for (int e = 0; e < per; ++e) {
                const float v = c[lane * per + e];
                b = fmaxf(b, fminf(a, v));
                a = fmaxf(a, v);
            }
            score = per > 1 ? a + b : a;
        }
        for (int k = 0; k < keep; ++k) {
            float bv = score;
            int bi = lane < n_groups ? lane : kMaxGroups + lane;
            wave_argmax(bv, bi);
            kept |= uint64_t(1) << (bi % kMaxGroups);
            if (lane == bi) score = -INFINITY;
        }
    }
    for (int k = 0; k < top; ++k) {
        float bv = -INFINITY;
        int bi = E;
        for (int e = lane; e < E; e += kWave) {
            const float v = ((kept >> (e / per)) & 1) || n_groups == 1 ? c[e] : -INFINITY;
            if (v > bv) {
                bv = v;
                bi = e;
            }
        }
        wave_argmax(bv, bi);
        const int best = min(bi, E - 1);
        if (lane == 0) {
            ids[k] = best < ra.n_listed ? best : -1;
            weights[k] = score(best) * ra.scale;
        }
        if (lane == best % kWave) c[best] = -INFINITY;
        wave_lds_order();
    }
    if (ra.extra && lane == 0) {
        ids[top] = ra.n_listed;
        weights[top] = 1.0f / (1.0f + expf(-z[E]));
    }
}

// The same for at most 64 outputs: an output a lane, its score in a register; zl is the lane's logit, and with `extra` lane 0 knows the
// token's own one. No trip through LDS. Groups of a power of two of outputs: their two largest meet in a butterfly, where a score that is no number brings the largest ahead
// of it in its group, which is what it leaves for the second largest in route_wave's order.
__device__ __forceinline__ void route_wave_lane(float zl, float own, const RouteArgs& ra, int E, int top, int* __restrict__ ids, float* __restrict__ weights) {
    const int lane = threadIdx.x % kWave;
    const bool real = lane < E, grouped = ra.keep < ra.n_groups;
    float s;
    if (ra.mode == 3) {
        const float v = real ? expf(zl - wave_max(real ? zl : -INFINITY)) : 0.0f;
        s = v * (1.0f / wave_sum(v));
    } else {
        s = 1.0f / (1.0f + expf(-zl));
    }
    float c = real ? s + (ra.correction != nullptr ? ra.correction[lane] : 0.0f) : -INFINITY;
    if (grouped) {
        const int per = E / ra.n_groups;
        float a = fmaxf(-INFINITY, c), b = -INFINITY;  // the two largest so far
        if (__builtin_amdgcn_ballot_w64(c != c) != 0) {
            float ahead = a;  // the largest up to this lane's, of its group
            for (int off = 1; off < per; off <<= 1) {
                const float before = __shfl_up(ahead, off, kWave);
                if (lane % per >= off) ahead = fmaxf(ahead, before);
            }
            if (c != c) b = ahead;
        }
        for (int off = 1; off < per; off <<= 1) {
            const float ao = __shfl_xor(a, off, kWave), bo = __shfl_xor(b, off, kWave);
            b = fmaxf(fminf(a, ao), fmaxf(b, bo));
            a = fmaxf(a, ao);
        }
        float score = __shfl(per > 1 ? a + b : a, (lane * per) % kWave, kWave);  // lane g: group g's
        if (lane >= ra.n_groups) score = -INFINITY;
        uint64_t kept = 0;
        for (int k = 0; k < ra.keep; ++k) {
            float bv = score;
            int bi = lane < ra.n_groups ? lane : kMaxGroups + lane;
            wave_argmax(bv, bi);
            kept |= uint64_t(1) << (bi % kMaxGroups);
            if (lane == bi) score = -INFINITY;
        }
        if (!(c > -INFINITY) || !((kept >> (lane / per)) & 1)) c = -INFINITY;
    }
    for (int k = 0; k < top; ++k) {
        float bv = c;
        int bi = grouped ? (c > -INFINITY ? lane : E) : real ? lane : kWave + lane;
        wave_argmax(bv, bi);
        const int best = min(bi, E - 1);
        if (lane == best) {
            ids[k] = best < ra.n_listed ? best : -1;
            weights[k] = s * ra.scale;
            c = -INFINITY;
        }
    }
    if (ra.extra && lane == 0) {
        ids[top] = ra.n_listed;
        weights[top] = 1.0f / (1.0f + expf(-own));
    }
}
__device__ __forceinline__ __host__ bool routes_in_lanes(const RouteArgs& ra, int E) {
    const int per = E / ra.n_groups;
    return E <= kWave && (ra.keep == ra.n_groups || (per & (per - 1)) == 0);
}

// a wave a token, four waves a workgroup
__global__ void __launch_bounds__(256)
moe_route_wave_kernel(const float* __restrict__ logits, int64_t ld, RouteArgs ra, int n, int E, int top, int* __restrict__ ids, float* __restrict__ weights) {
    extern __shared__ int sh[];
    const int wave = threadIdx.x / kWave, t = blockIdx.x * 4 + wave;
    if (t >= n) return;
    const int64_t at = static_cast<int64_t>(t) * (top + ra.extra);
    if (routes_in_lanes(ra, E)) {
        const float* z = logits + static_cast<int64_t>(t) * ld;
        route_wave_lane(z[min(static_cast<int>(threadIdx.x) % kWave, E - 1)], z[ra.extra ? E : 0], ra, E, top, ids + at, weights + at);
        return;
    }
    route_wave(logits + static_cast<int64_t>(t) * ld, ra, E, top, ids + at, weights + at, reinterpret_cast<float*>(sh) + wave * E);
}

// mode 0: the largest logits, softmax over the chosen ones; mode 1: softmax over all, groups, weights by their sum
__device__ __forceinline__ void route_any(const float* __restrict__ z, int E, int top, int mode, int n_groups, int keep, int* __restrict__ ids,
                                          float* __restrict__ weights) {
    if (mode == 1) route_token_groups(z, E, top, n_groups, keep, ids, weights);
    else route_token(z, E, top, ids, weights);
}

__global__ void __launch_bounds__(256)
moe_route_kernel(const float* __restrict__ logits, int64_t ld, int n, int E, int top, int* __restrict__ ids, float* __restrict__ weights,
                 int mode, int n_groups, int keep) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= n) return;
    route_any(logits + static_cast<int64_t>(t) * ld, E, top, mode, n_groups, keep, ids + static_cast<int64_t>(t) * top, weights + static_cast<int64_t>(t) * top);
}

// The entries of `ids` listed by expert in tiles of `block` places; one workgroup of 1,024 threads runs this.
__device__ __forceinline__ void align_entries(const int* __restrict__ ids, int n_entries, int E, int block, int* __restrict__ rows_list,
                                              int* __restrict__ tile_group, int max_tiles, int* sh) {
    int* counts = sh;     // [E]
    int* first = sh + E;  // [E + 1]: the first place of each expert
    const int tid = threadIdx.x;
    for (int e = tid; e < E; e += 1024) counts[e] = 0;
    for (int i = tid; i < max_tiles * block; i += 1024) rows_list[i] = -1;
    for (int i = tid; i < max_tiles; i += 1024) tile_group[i] = -1;
    __syncthreads();
    for (int i = tid; i < n_entries; i += 1024) {
        const int e = ids[i];
        if (e >= 0 && e < E) atomicAdd(&counts[e], 1);
    }
    __syncthreads();
    if (tid == 0) {
        int at = 0;
        for (int e = 0; e < E; ++e) {
            first[e] = at;
            const int tiles = (counts[e] + block - 1) / block;
            for (int i = 0; i < tiles; ++i)
                if (at / block + i < max_tiles) tile_group[at / block + i] = e;
            at += tiles * block;
            counts[e] = 0;  // counts the entries placed so far from here on
        }
        first[E] = at;
    }
    __syncthreads();
    for (int i = tid; i < n_entries; i += 1024) {
        const int e = ids[i];
        if (e < 0 || e >= E) continue;
        const int place = first[e] + atomicAdd(&counts[e], 1);
        if (place < max_tiles * block) rows_list[place] = i;
    }
}

__global__ void __launch_bounds__(1024)
moe_align_kernel(const int* __restrict__ ids, int n_entries, int E, int block, int* __restrict__ rows_list, int* __restrict__ tile_group,
                 int max_tiles) {
    extern __shared__ int sh[];
    align_entries(ids, n_entries, E, block, rows_list, tile_group, max_tiles, sh);
}

// route_token by a wave, an expert a lane: the same choices (a NaN counts as the lowest, unless it is the first that is left) and the same bits.
__device__ __forceinline__ void route_wave_softmax(float zl, int E, int top, int* __restrict__ ids, float* __restrict__ weights) {
    const int lane = threadIdx.x % kWave;
    const uint32_t u = __float_as_uint(zl + 0.0f);  // (one zero)
    uint32_t key = lane >= E ? 0u : zl != zl ? 1u : (u & 0x80000000u) ? ~u : u | 0x80000000u;  // 0: not there, or taken
    const uint64_t nans = __builtin_amdgcn_ballot_w64(zl != zl && lane < E);
    int chosen = 0;
    float value = 0.0f;  // lane k: the k-th choice
    for (int k = 0; k < top; ++k) {
        uint32_t bk = key;
        int best = lane;
        wave_argmax(bk, best);
        const int first = __builtin_ctzll(__builtin_amdgcn_ballot_w64(key != 0));
        if ((nans >> first) & 1) best = first;
        const float v = lane_of(zl, __builtin_amdgcn_readfirstlane(best));
        if (lane == k) {
            chosen = best;
            value = v;
        }
        if (lane == best) key = 0;
    }
    const float e = lane < top ? expf(value - lane_of(value, 0)) : 0.0f;
    float sum = 0.0f;
    for (int k = 0; k < top; ++k) sum += lane_of(e, k);
    if (lane < top) {
        ids[lane] = chosen;
        weights[lane] = e / sum;
    }
}

// Mode 0 for steps of more tokens: a wave a token, four a workgroup, while there are few tokens for what a thread would have to scan one after the other (us with
// the lists, a thread / a wave a token: 2 of 8 experts 1,640 tokens 11.8 / 10.0, 8,000 26.8 / 26.9, 20,000 55.8 / 59.0; 1 of 2 1,025 6.1 / 6.3, 16,000 30.9 / 34.0;
// 2 of 2 2,000 11.2 / 11.1, 8,000 30.1 / 31.9; 2 of 16 16,000 50.6 / 50.5; 8 of 64 5,000 386 / 73).
bool waves_route(int n, int E, int top) { return E > 1 && E <= kWave && n <= int64_t(512) * E * top; }

__global__ void __launch_bounds__(256)
moe_route_softmax_kernel(const float* __restrict__ logits, int64_t ld, int n, int E, int top, int* __restrict__ ids, float* __restrict__ weights) {
    const int t = blockIdx.x * 4 + threadIdx.x / kWave;
    if (t >= n) return;
    const int64_t at = static_cast<int64_t>(t) * top;
    route_wave_softmax(logits[static_cast<int64_t>(t) * ld + min(static_cast<int>(threadIdx.x) % kWave, E - 1)], E, top, ids + at, weights + at);
}

// Choices (modes 0, 2 and 3) and lists of a step of at most kWaveRouteTokens tokens, few experts and entries (a decoding step): one workgroup, whose time is the trips of
// what one thread writes and another reads. A wave chooses for a token, an expert a lane; ids, counts and lists stay in LDS, every wave sums up the experts'
// first places by itself, an expert a lane, and everything leaves once at the end. (The kernel below has a thread choose, or a wave with its scores in LDS, clears the lists in memory,
// reads the ids back from there twice and has one thread lay out the tiles: 4 tokens, 2 of 8 experts
// 6.7 -> 4.9 us, 8 of 64 235 -> 17.5; with the product ahead, a layer's step of 4 tokens at GPT-2 small's width gains 4.1 us with groups of experts, 3.1 with softmax scores over
// all, 1.0 with the largest logits, the last two of whose choices were as short before.)
constexpr int kSmallExperts = 64, kSmallEntries = 1024, kSmallPlaces = 4096;

// The router's own product ahead of that, for up to 16 tokens and outputs: the logits are one strip of gemm_skinny.hip's streaming kernel, one workgroup, and this one takes it
// over with that kernel's waves, order of sums and bits. K: whole units of 64; 1 << split_shift waves share it, two units a trip.
struct RouterProduct {
    const bf16_t* a;
    int64_t lda;
    const bf16_t* w;
    const float* bias;
    int columns, K, split_shift;
    float* logits;
};
typedef __attribute__((ext_vector_type(8))) __bf16 moe_bf16x8;
typedef __attribute__((ext_vector_type(4))) float moe_f32x4;
constexpr int kRouterSide = 16;

template <bool PRODUCT>
__global__ void __launch_bounds__(1024)
moe_route_align_small_kernel(const float* __restrict__ logits, int64_t ld, int n, int E, int top, int* __restrict__ ids, float* __restrict__ weights,
                             int block, int* __restrict__ rows_list, int* __restrict__ tile_group, int max_tiles, RouteArgs ra, RouterProduct rp) {
    extern __shared__ int list[];  // [places]
    __shared__ int ids_of[kSmallEntries], counts[kSmallExperts];
    __shared__ float weights_of[kSmallEntries];
    const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t / kWave), lane = t % kWave, each = top + ra.extra, entries = n * each, places = max_tiles * block;
    constexpr int kEach = kWaveRouteTokens / (1024 / kWave);  // tokens a wave: all their logits are asked for together
    float zl[kEach], own[kEach];
    if constexpr (PRODUCT) {
        __shared__ float sums[1024 / kWave][kRouterSide * kRouterSide], z[kRouterSide][kRouterSide];
        const int i = lane % 16, g = lane / 16, splits = 1 << rp.split_shift, units = rp.K / 64, trips = (units + 1) / 2;
        const int live = min(splits, trips);
        if (wave < live) {
            const bf16_t* const w = rp.w + static_cast<int64_t>(min(i, rp.columns - 1)) * rp.K + g * 8;
            const bf16_t* const a = rp.a + static_cast<int64_t>(min(i, n - 1)) * rp.lda + g * 8;
            moe_f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
            for (int trip = wave; trip < trips; trip += splits) {
                moe_bf16x8 x[4], y[4];
#pragma unroll
                for (int h = 0; h < 4; ++h) {
                    const int k = min(trip * 128 + 32 * h, rp.K - 32);  // (a unit past the end: read and not multiplied)
                    x[h] = *reinterpret_cast<const moe_bf16x8*>(w + k);
                    y[h] = *reinterpret_cast<const moe_bf16x8*>(a + k);
                }
#pragma unroll
                for (int h = 0; h < 4; ++h)
                    if (h < 2 || 2 * trip + 1 < units) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[h], y[h], acc, 0, 0, 0);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) sums[wave][i * 16 + 4 * g + r] = acc[r];
        }
        for (int q = t; q < places; q += 1024) list[q] = -1;
        if (t < kSmallExperts) counts[t] = 0;
        const int m = t / 16, c = t % 16;
        const bool mine = t < 256 && m < n && c < rp.columns;
        const float bias = rp.bias != nullptr ? rp.bias[min(c, rp.columns - 1)] : 0.0f;
        lds_barrier();
        if (mine) {
            float v = 0.0f;
            for (int q = 0; q < live; ++q) v += sums[q][t];
            v += bias;
            z[m][c] = v;
            rp.logits[static_cast<int64_t>(m) * ld + c] = v;
        }
        lds_barrier();
        zl[0] = z[min(wave, n - 1)][min(lane, E - 1)];
        own[0] = z[min(wave, n - 1)][ra.extra ? E : 0];
    } else {
#pragma unroll
        for (int j = 0; j < kEach; ++j) {
            const float* const z = logits + static_cast<int64_t>(min(wave + j * (1024 / kWave), n - 1)) * ld;
            zl[j] = z[min(lane, E - 1)];
            own[j] = z[ra.extra ? E : 0];
        }
        for (int i = t; i < places; i += 1024) list[i] = -1;
        if (t < kSmallExperts) counts[t] = 0;
    }
#pragma unroll
    for (int j = 0; j < (PRODUCT ? 1 : kEach); ++j) {
        const int i = wave + j * (1024 / kWave);
        if (i >= n) continue;
        if (ra.mode == 0) route_wave_softmax(zl[j], E, top, ids_of + i * each, weights_of + i * each);
        else route_wave_lane(zl[j], own[j], ra, E, top, ids_of + i * each, weights_of + i * each);
    }
    lds_barrier();
    int e = -1, rank = 0;
    if (t < entries) {
        e = ids_of[t];
        ids[t] = e;
        weights[t] = weights_of[t];
        if (e >= 0) rank = atomicAdd(&counts[e], 1);
    }
    lds_barrier();
    const int tiles = (counts[lane] + block - 1) / block;  // of expert `lane` (past the experts: none)
    int up_to = tiles;
    for (int off = 1; off < kWave; off <<= 1) {
        const int before = __shfl_up(up_to, off, kWave);
        if (lane >= off) up_to += before;
    }
    const int at = up_to - tiles, used = __shfl(up_to, kWave - 1, kWave), place = __shfl(at, max(e, 0), kWave) * block + rank;
    if (e >= 0 && place < places) list[place] = t;
    if (wave == 0) {
        for (int i = at; i < min(up_to, max_tiles); ++i) tile_group[i] = lane;
        for (int i = used + lane; i < max_tiles; i += kWave) tile_group[i] = -1;
    }
    lds_barrier();
    for (int i = t; i < places; i += 1024) rows_list[i] = list[i];
}

// Both in one launch for steps of at most 1,024 tokens: a thread routes a token, then the workgroup lists the entries.
__global__ void __launch_bounds__(1024)
moe_route_align_kernel(const float* __restrict__ logits, int64_t ld, int n, int E, int top, int* __restrict__ ids, float* __restrict__ weights,
                       int block, int* __restrict__ rows_list, int* __restrict__ tile_group, int max_tiles, RouteArgs ra) {
    extern __shared__ int sh[];
    const int t = threadIdx.x;
    if (ra.mode >= 2) {  // a wave a token, sixteen at a time
        const int wave = t / kWave;
        if (routes_in_lanes(ra, E)) {
            constexpr int kEach = kWaveRouteTokens / (1024 / kWave);  // tokens a wave: all their logits are asked for together
            float zl[kEach], own[kEach];
#pragma unroll
            for (int j = 0; j < kEach; ++j) {
                const float* z = logits + static_cast<int64_t>(min(wave + j * (1024 / kWave), n - 1)) * ld;
                zl[j] = z[min(t % kWave, E - 1)];
                own[j] = z[ra.extra ? E : 0];
            }
#pragma unroll
            for (int j = 0; j < kEach; ++j) {
                const int i = wave + j * (1024 / kWave);
                const int64_t at = static_cast<int64_t>(i) * (top + ra.extra);
                if (i < n) route_wave_lane(zl[j], own[j], ra, E, top, ids + at, weights + at);
            }
        } else for (int i = wave; i < n; i += 1024 / kWave) {
            const int64_t at = static_cast<int64_t>(i) * (top + ra.extra);
            route_wave(logits + static_cast<int64_t>(i) * ld, ra, E, top, ids + at, weights + at, reinterpret_cast<float*>(sh) + wave * E);
        }
    } else if (t < n) route_any(logits + static_cast<int64_t>(t) * ld, E, top, ra.mode, ra.n_groups, ra.keep, ids + static_cast<int64_t>(t) * top, weights + static_cast<int64_t>(t) * top);
    __syncthreads();  // (the ids are read back by other threads of this workgroup)
    align_entries(ids, n * (top + ra.extra), ra.n_listed + ra.extra, block, rows_list, tile_group, max_tiles, sh);
}

}  // namespace liyab

using namespace liyab;

// ids and weights: [n, top + extra]. n_listed, extra: see the head of this file (n_experts and 0 outside modes 2 and 3).
extern "C" int liyab_moe_route(const float* logits, int64_t ld, int n, int n_experts, int top, int* ids, float* weights, int mode, int n_groups,
                               int keep, const float* correction, float scale, int n_listed, int extra, hipStream_t stream) {
    LIYAB_REQUIRE(logits && ids && weights, "moe_route: null pointer");
    LIYAB_REQUIRE(mode == 0 || (mode >= 1 && mode <= 3 && n_groups >= 1 && n_groups <= kMaxGroups && n_experts % n_groups == 0 && keep >= 1 && keep <= n_groups &&
                                top <= keep * (n_experts / n_groups)),
                  "moe_route: %d of %d groups of %d experts do not hold %d choices (at most %d groups)", keep, n_groups, n_experts, top, kMaxGroups);
    LIYAB_REQUIRE(n >= 0 && n_experts > 0 && top >= 1 && top <= n_experts && top <= kMaxTop && ld >= n_experts,
                  "moe_route: bad sizes n=%d experts=%d top=%d (at most %d choices a token)", n, n_experts, top, kMaxTop);
    LIYAB_REQUIRE(mode < 2 || n_experts <= kMaxWaveExperts, "moe_route: %d experts; at most %d are taken in this mode", n_experts, kMaxWaveExperts);
    LIYAB_REQUIRE(n_listed >= 1 && n_listed <= n_experts && (extra == 0 || extra == 1) && (mode >= 2 || (n_listed == n_experts && extra == 0)) && ld >= n_experts + extra,
                  "moe_route: %d listed of %d outputs, %d entries for every token do not go with this mode", n_listed, n_experts, extra);
    if (n == 0) return 0;
    if (mode == 0 && waves_route(n, n_experts, top)) {
        moe_route_softmax_kernel<<<(n + 3) / 4, 256, 0, stream>>>(logits, ld, n, n_experts, top, ids, weights);
        return check_launch("moe_route");
    }
    if (mode >= 2) {
        const RouteArgs ra{mode, n_groups, keep, correction, scale, n_listed, extra};
        moe_route_wave_kernel<<<(n + 3) / 4, 256, 4 * n_experts * sizeof(float), stream>>>(logits, ld, ra, n, n_experts, top, ids, weights);
        return check_launch("moe_route");
    }
    moe_route_kernel<<<(n + 255) / 256, 256, 0, stream>>>(logits, ld, n, n_experts, top, ids, weights, mode, n_groups, keep);
    return check_launch("moe_route");
}

extern "C" int liyab_moe_align(const int* ids, int n_entries, int n_experts, int block, int* rows_list, int* tile_group, int max_tiles,
                               hipStream_t stream) {
    LIYAB_REQUIRE(ids && rows_list && tile_group, "moe_align: null pointer");
    LIYAB_REQUIRE(n_entries >= 0 && n_experts > 0 && n_experts <= 4096 && block > 0, "moe_align: bad sizes (at most 4,096 experts)");
    LIYAB_REQUIRE(static_cast<int64_t>(max_tiles) * block >= static_cast<int64_t>(n_entries) + static_cast<int64_t>(n_entries < n_experts ? n_entries : n_experts) * (block - 1),
                  "moe_align: %d tiles of %d places do not hold %d entries of %d experts", max_tiles, block, n_entries, n_experts);
    if (n_entries == 0) return 0;
    moe_align_kernel<<<1, 1024, (2 * n_experts + 1) * sizeof(int), stream>>>(ids, n_entries, n_experts, block, rows_list, tile_group, max_tiles);
    return check_launch("moe_align");
}

// `rp`: the router's product ahead of the choice (or null).
static int route_align(const RouterProduct* rp, const float* logits, int64_t ld, int n, int n_experts, int top, int* ids, float* weights, int block,
                                     int* rows_list, int* tile_group, int max_tiles, int mode, int n_groups, int keep, const float* correction,
                                     float scale, int n_listed, int extra, hipStream_t stream) {
    LIYAB_REQUIRE(n <= 1024, "moe_route_align: %d tokens; one workgroup routes at most 1,024 (moe_route and moe_align take more)", n);
    if (const int rc = liyab_moe_route(logits, ld, 0, n_experts, top, ids, weights, mode, n_groups, keep, correction, scale, n_listed, extra, stream)) return rc;  // (the checks of both,
    const int listed = n_listed + extra;
    if (const int rc = liyab_moe_align(ids, 0, listed, block, rows_list, tile_group, max_tiles, stream)) return rc;    //  nothing launched)
    LIYAB_REQUIRE(n >= 0 && static_cast<int64_t>(max_tiles) * block >= static_cast<int64_t>(n) * (top + extra) + static_cast<int64_t>(n * (top + extra) < listed ? n * (top + extra) : listed) * (block - 1),
                  "moe_route_align: %d tiles of %d places do not hold %d entries of %d experts", max_tiles, block, n * (top + extra), listed);
    LIYAB_REQUIRE(mode < 2 || (n <= kWaveRouteTokens && n_experts <= 512), "moe_route_align: %d tokens of %d experts; modes 2 and 3 take %d of 512 here", n, n_experts, kWaveRouteTokens);
    if (n == 0) return 0;
    const size_t smem = sizeof(int) * (mode >= 2 ? (1024 / kWave) * static_cast<size_t>(n_experts) + 4 : 2 * static_cast<size_t>(n_experts) + 1);  // (the scores; then the lists' counts)
    const RouteArgs ra{mode, n_groups, keep, correction, scale, n_listed, extra};
    // More than a token a wave and few experts: a thread a token is faster (64 tokens, 2 of 8 experts 7.2 us against 10.6; 8 of 64 246 against 36), and from some
    // ten tokens on where it has little to scan (16 tokens, 1 of 2 3.3 against 3.7, 1 of 4 3.8 and 4.1, 2 of 4 5.0 and 4.8; 8 tokens, 1 of 2 3.3 and 3.3).
    const int64_t places = static_cast<int64_t>(max_tiles) * block;
    const bool small = n <= kWaveRouteTokens && n_experts > 1 && n_experts <= kSmallExperts && listed <= kSmallExperts && n * (top + extra) <= kSmallEntries && places <= kSmallPlaces;
    if (small && (mode == 0 ? n <= 8 || (n <= 1024 / kWave && n_experts * top > 4) || n_experts * top > 64 : mode >= 2 && routes_in_lanes(ra, n_experts))) {
        if (rp != nullptr)
            moe_route_align_small_kernel<true><<<1, 1024, static_cast<size_t>(places) * sizeof(int), stream>>>(logits, ld, n, n_experts, top, ids, weights, block, rows_list, tile_group, max_tiles, ra, *rp);
        else
            moe_route_align_small_kernel<false><<<1, 1024, static_cast<size_t>(places) * sizeof(int), stream>>>(logits, ld, n, n_experts, top, ids, weights, block, rows_list, tile_group, max_tiles, ra, RouterProduct{});
        return check_launch("moe_route_align");
    }
    LIYAB_REQUIRE(rp == nullptr, "moe_router: %d tokens of %d experts are not taken with the router's product", n, n_experts);
    moe_route_align_kernel<<<1, 1024, smem, stream>>>(logits, ld, n, n_experts, top, ids, weights, block, rows_list, tile_group, max_tiles, ra);
    return check_launch("moe_route_align");
}

extern "C" int liyab_moe_route_align(const float* logits, int64_t ld, int n, int n_experts, int top, int* ids, float* weights, int block,
                                     int* rows_list, int* tile_group, int max_tiles, int mode, int n_groups, int keep, const float* correction,
                                     float scale, int n_listed, int extra, hipStream_t stream) {
    return route_align(nullptr, logits, ld, n, n_experts, top, ids, weights, block, rows_list, tile_group, max_tiles, mode, n_groups, keep, correction, scale, n_listed, extra, stream);
}

// The same behind the router's product, logits = a . w^T + bias for a [n <= 16, K] and w [columns <= 16, K] in bfloat16, K whole units of 64 and not of 16,384: the logits of
// liyab_gemm_skinny, bit for bit, whose launch goes. columns: n_experts, or more (of which the choice sees the first n_experts and, with `extra`, the one behind them).
extern "C" int liyab_moe_router(const void* a, int64_t lda, const void* w, const float* bias, int columns, int K, float* logits, int64_t ld, int n, int n_experts, int top, int* ids,
                                float* weights, int block, int* rows_list, int* tile_group, int max_tiles, int mode, int n_groups, int keep, const float* correction, float scale,
                                int n_listed, int extra, hipStream_t stream) {
    LIYAB_REQUIRE(a && w, "moe_router: null operand");
    LIYAB_REQUIRE(n <= kRouterSide && columns <= kRouterSide && columns >= n_experts + extra && ld >= columns && K > 0 && K % 64 == 0 && K % 16384 != 0 && lda >= K && lda % 8 == 0,
                  "moe_router: bad sizes n=%d columns=%d of %d experts K=%d", n, columns, n_experts, K);
    LIYAB_REQUIRE((reinterpret_cast<uintptr_t>(a) & 15) == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0, "moe_router: operands must be 16-byte aligned");
    int split_shift = 0;  // the waves that gemm_skinny.hip's choice has for one strip (choose_ksplit)
    while (split_shift < 4 && K / 64 > (2 << split_shift)) ++split_shift;
    const RouterProduct rp{static_cast<const bf16_t*>(a), lda, static_cast<const bf16_t*>(w), bias, columns, K, split_shift, logits};
    return route_align(&rp, logits, ld, n, n_experts, top, ids, weights, block, rows_list, tile_group, max_tiles, mode, n_groups, keep, correction, scale, n_listed, extra, stream);
}
