// The residual stream as several copies that learned weights mix (hyper-connections), or as one: the rows' update between two
// sublayers, together with what the next sublayer reads.
//
// liyab_streams_update, for each token (its S streams of d 32-bit floats lie side by side in x):
//   y    = the sum of the sublayer's n_sum rows of the token, in their order; where `ids` says -1 for one of the first n_ids of
//          them (a routed feed-forward's entry that took an identity expert), weights * h takes the place of a row: h are the rows the
//          sublayer read (they may lie where `out` goes: a thread reads its entries of them before it writes)
//   x_t <- sum_s mix[s, t] x_s + add[t] y          all streams from the old ones; without `mix`: x_t + add[t] y; without `add`: ones
//   u    = sum_s in[s] x_s of the new streams (without `in`: their plain sum)
//   out  = u / sqrt(mean(u^2) + eps) * w in the output type
// Every part is optional: `enter` (rows [n, d]) first sets all streams to those rows; without y the streams stay as they are;
// without `out` nothing is read off them; `rows` gathers (what is read off them only: the final norm of the wanted rows).
// All sums and the norm are 32-bit; a result is rounded once, to the output type.
#include "common.h"
#include "launchers.h"

namespace liyab {

constexpr int ST_THREADS = 256;
constexpr int ST_MAX_STREAMS = 8;
constexpr int ST_HELD = 4;  // groups of VEC entries of u a thread keeps between the two passes; wider rows are read again

struct StreamsArgs {
    float* x;
    const float* enter;
    const float* y;
    int n_sum, n_ids;
    const int* ids;
    const float* weights;
    const void* h;
    const float *mix, *add, *in, *w;
    float eps;
    void* out;
    const int* rows;
    int d;
};

template <int VEC>
struct StVec {
    float v[VEC];
};
template <int VEC>
__device__ __forceinline__ StVec<VEC> st_load(const float* p) {
    StVec<VEC> r;
    if constexpr (VEC == 4) {
        const f32x4_t q = *reinterpret_cast<const f32x4_t*>(p);
        r.v[0] = q[0]; r.v[1] = q[1]; r.v[2] = q[2]; r.v[3] = q[3];
    } else {
        r.v[0] = *p;
    }
    return r;
}

template <typename T, int S, int VEC>
__global__ void __launch_bounds__(ST_THREADS)
streams_update_kernel(StreamsArgs a) {
    __shared__ float red[ST_THREADS / kWave];
    const int t = blockIdx.x, d = a.d;
    const int64_t src = a.rows != nullptr ? a.rows[t] : t;
    float* xr = a.x + src * S * d;
    float mix[S][S], add[S], in[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        add[s] = a.add != nullptr ? a.add[s] : 1.0f;
        in[s] = a.in != nullptr ? a.in[s] : 1.0f;
#pragma unroll
        for (int to = 0; to < S; ++to) mix[s][to] = a.mix != nullptr ? a.mix[s * S + to] : (s == to ? 1.0f : 0.0f);
    }
    const int groups = d / VEC;  // (VEC 4 only where d is a multiple of 4)
    auto streams_of = [&](int i, StVec<VEC> (&x)[S]) {
        if (a.enter != nullptr) {
            const StVec<VEC> e = st_load<VEC>(a.enter + src * d + i);
#pragma unroll
            for (int s = 0; s < S; ++s) x[s] = e;
        } else {
#pragma unroll
            for (int s = 0; s < S; ++s) x[s] = st_load<VEC>(xr + static_cast<int64_t>(s) * d + i);
        }
    };
    auto read_off = [&](const StVec<VEC> (&x)[S]) {
        StVec<VEC> u;
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            float v = in[0] * x[0].v[e];
#pragma unroll
            for (int s = 1; s < S; ++s) v = fmaf(in[s], x[s].v[e], v);
            u.v[e] = v;
        }
        return u;
    };
    // the new streams at entries i .. i + VEC - 1, written where they changed; what the next sublayer reads of them
    auto update = [&](int i) {
        StVec<VEC> x[S];
        streams_of(i, x);
        if (a.y != nullptr) {
            const float* yr = a.y + src * a.n_sum * d + i;
            StVec<VEC> y;
#pragma unroll
            for (int e = 0; e < VEC; ++e) y.v[e] = 0.0f;
            for (int k = 0; k < a.n_sum; ++k) {
                if (k < a.n_ids && a.ids[src * a.n_ids + k] < 0) {  // (the same for the whole workgroup)
                    const float weight = a.weights[src * a.n_ids + k];
                    const T* h = static_cast<const T*>(a.h) + src * d + i;
#pragma unroll
                    for (int e = 0; e < VEC; ++e) y.v[e] = fmaf(weight, to_float<T>(h[e]), y.v[e]);
                } else {
                    const StVec<VEC> r = st_load<VEC>(yr + static_cast<int64_t>(k) * d);
#pragma unroll
                    for (int e = 0; e < VEC; ++e) y.v[e] += r.v[e];
                }
            }
            StVec<VEC> z[S];
#pragma unroll
            for (int to = 0; to < S; ++to)
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    float v = add[to] * y.v[e];
#pragma unroll
                    for (int s = 0; s < S; ++s) v = fmaf(mix[s][to], x[s].v[e], v);
                    z[to].v[e] = v;
                }
#pragma unroll
            for (int s = 0; s < S; ++s) x[s] = z[s];
        }
        if (a.y != nullptr || a.enter != nullptr) {
#pragma unroll
            for (int s = 0; s < S; ++s) {
                if constexpr (VEC == 4) store4<float>(xr + static_cast<int64_t>(s) * d + i, x[s].v);
                else xr[static_cast<int64_t>(s) * d + i] = x[s].v[0];
            }
        }
        return read_off(x);
    };
    StVec<VEC> held[ST_HELD];
    float ss = 0.0f;
#pragma unroll
    for (int j = 0; j < ST_HELD; ++j) {
        const int g = threadIdx.x + j * ST_THREADS;
        if (g < groups) {
            held[j] = update(g * VEC);
#pragma unroll
            for (int e = 0; e < VEC; ++e) ss = fmaf(held[j].v[e], held[j].v[e], ss);
        }
    }
    for (int g = threadIdx.x + ST_HELD * ST_THREADS; g < groups; g += ST_THREADS) {
        const StVec<VEC> u = update(g * VEC);
#pragma unroll
        for (int e = 0; e < VEC; ++e) ss = fmaf(u.v[e], u.v[e], ss);
    }
    if (a.out == nullptr) return;
    ss = wave_sum(ss);
    if (threadIdx.x % kWave == 0) red[threadIdx.x / kWave] = ss;
    __syncthreads();
    float total = 0.0f;
#pragma unroll
    for (int i = 0; i < ST_THREADS / kWave; ++i) total += red[i];
    const float scale = 1.0f / sqrtf(total / static_cast<float>(d) + a.eps);
    T* o = static_cast<T*>(a.out) + static_cast<int64_t>(t) * d;
    auto finish = [&](int i, const StVec<VEC>& u) {
        float v[VEC];
#pragma unroll
        for (int e = 0; e < VEC; ++e) v[e] = u.v[e] * scale;
        if (a.w != nullptr) {
            const StVec<VEC> w = st_load<VEC>(a.w + i);
#pragma unroll
            for (int e = 0; e < VEC; ++e) v[e] *= w.v[e];
        }
        if constexpr (VEC == 4) store4<T>(o + i, v);
        else o[i] = from_float<T>(v[0]);
    };
#pragma unroll
    for (int j = 0; j < ST_HELD; ++j) {
        const int g = threadIdx.x + j * ST_THREADS;
        if (g < groups) finish(g * VEC, held[j]);
    }
    for (int g = threadIdx.x + ST_HELD * ST_THREADS; g < groups; g += ST_THREADS) {
        StVec<VEC> x[S];
#pragma unroll
        for (int s = 0; s < S; ++s) x[s] = st_load<VEC>(xr + static_cast<int64_t>(s) * d + g * VEC);  // (each thread reads what it wrote)
        finish(g * VEC, read_off(x));
    }
}

// The same for rows of up to 1,024 (a multiple of 4) and a sublayer of up to four rows a token: a group of 4 entries a thread. The kernel is a link of a decode
// step's chain, two of them a layer, and waits for memory and for its own instructions: everything it reads is asked for together, the norm's weight too,
// with no load under a branch (what is not given is read from the streams and dropped), and nothing is there that it does not run (IDS: identity experts).
// us, a step of 4 tokens of 2 x 768 in a chain, before / now: 2.8 / 2.6, with two rows a token 3.0 / 2.6, three 3.1 / 2.6, with identity experts 3.2 / 2.9. The same
// operations, the same bits.
template <typename T, int S, bool IDS>
__global__ void __launch_bounds__(ST_THREADS)
streams_row_kernel(StreamsArgs a) {
    constexpr int SUM = 4;
    __shared__ float red[ST_THREADS / kWave];
    const int t = blockIdx.x, d = a.d, groups = d / 4;
    const int64_t src = a.rows != nullptr ? a.rows[t] : t;
    float* const xr = a.x + src * S * d;
    const bool mine = threadIdx.x < groups;
    const int i = min(static_cast<int>(threadIdx.x), groups - 1) * 4;  // (past the row: its last group again, dropped)
    const float* const nothing = xr;
    const float *const mix_at = a.mix != nullptr ? a.mix : nothing, *const add_at = a.add != nullptr ? a.add : nothing, *const in_at = a.in != nullptr ? a.in : nothing;
    float mix[S][S], add[S], in[S];
    StVec<4> x[S], r[SUM], w;
#pragma unroll
    for (int s = 0; s < S; ++s) x[s] = st_load<4>(a.enter != nullptr ? a.enter + src * d + i : xr + static_cast<int64_t>(s) * d + i);
#pragma unroll
    for (int k = 0; k < SUM; ++k) r[k] = st_load<4>(a.y != nullptr ? a.y + (src * a.n_sum + min(k, a.n_sum - 1)) * d + i : nothing + i);
    w = st_load<4>((a.w != nullptr ? a.w : nothing) + i);
#pragma unroll
    for (int s = 0; s < S; ++s) {
        add[s] = add_at[s];
        in[s] = in_at[s];
#pragma unroll
        for (int to = 0; to < S; ++to) mix[s][to] = mix_at[s * S + to];
    }
    int id[SUM];
    float weight[SUM], h[4];
    if constexpr (IDS) {
        const T* const rows = static_cast<const T*>(a.h) + src * d + i;
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = to_float<T>(rows[e]);
#pragma unroll
        for (int k = 0; k < SUM; ++k) {
            id[k] = a.ids[src * a.n_ids + min(k, a.n_ids - 1)];
            weight[k] = a.weights[src * a.n_ids + min(k, a.n_ids - 1)];
        }
    }
    // (loaded values from here on: no load is drawn into the choices below)
#pragma unroll
    for (int k = 0; k < SUM; ++k) settle_loads(r[k].v);
#pragma unroll
    for (int s = 0; s < S; ++s) settle_loads(x[s].v);
    settle_loads(w.v);
    if constexpr (IDS) settle_loads(h);
#pragma unroll
    for (int s = 0; s < S; ++s) {
        if (a.add == nullptr) add[s] = 1.0f;
        if (a.in == nullptr) in[s] = 1.0f;
#pragma unroll
        for (int to = 0; to < S; ++to)
            if (a.mix == nullptr) mix[s][to] = s == to ? 1.0f : 0.0f;
    }
    if (a.y != nullptr) {
        float y[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < SUM; ++k) {
            if (k >= a.n_sum) break;
            const bool identity = IDS && k < a.n_ids && id[k] < 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] = identity ? fmaf(weight[k], h[e], y[e]) : y[e] + r[k].v[e];
        }
        StVec<4> z[S];
#pragma unroll
        for (int to = 0; to < S; ++to)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float v = add[to] * y[e];
#pragma unroll
                for (int s = 0; s < S; ++s) v = fmaf(mix[s][to], x[s].v[e], v);
                z[to].v[e] = v;
            }
#pragma unroll
        for (int s = 0; s < S; ++s) x[s] = z[s];
    }
    if ((a.y != nullptr || a.enter != nullptr) && mine) {
#pragma unroll
        for (int s = 0; s < S; ++s) store4<float>(xr + static_cast<int64_t>(s) * d + i, x[s].v);
    }
    if (a.out == nullptr) return;
    float u[4], ss = 0.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float v = in[0] * x[0].v[e];
#pragma unroll
        for (int s = 1; s < S; ++s) v = fmaf(in[s], x[s].v[e], v);
        u[e] = v;
        ss = fmaf(v, v, ss);
    }
    ss = wave_sum(mine ? ss : 0.0f);
    if (threadIdx.x % kWave == 0) red[threadIdx.x / kWave] = ss;
    lds_barrier();
    float total = 0.0f;
#pragma unroll
    for (int j = 0; j < ST_THREADS / kWave; ++j) total += red[j];
    const float scale = 1.0f / sqrtf(total / static_cast<float>(d) + a.eps);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        u[e] *= scale;
        if (a.w != nullptr) u[e] *= w.v[e];
    }
    if (mine) store4<T>(static_cast<T*>(a.out) + static_cast<int64_t>(t) * d + i, u);
}

template <typename T, bool IDS>
bool launch_streams_row(const StreamsArgs& a, int n, int S, hipStream_t stream) {
    switch (S) {
        case 1: streams_row_kernel<T, 1, IDS><<<n, ST_THREADS, 0, stream>>>(a); return true;
        case 2: streams_row_kernel<T, 2, IDS><<<n, ST_THREADS, 0, stream>>>(a); return true;
        case 3: streams_row_kernel<T, 3, IDS><<<n, ST_THREADS, 0, stream>>>(a); return true;
        case 4: streams_row_kernel<T, 4, IDS><<<n, ST_THREADS, 0, stream>>>(a); return true;
        default: return false;
    }
}

template <typename T, int VEC>
void launch_streams(const StreamsArgs& a, int n, int S, hipStream_t stream) {
    switch (S) {
        case 1: streams_update_kernel<T, 1, VEC><<<n, ST_THREADS, 0, stream>>>(a); break;
        case 2: streams_update_kernel<T, 2, VEC><<<n, ST_THREADS, 0, stream>>>(a); break;
        case 3: streams_update_kernel<T, 3, VEC><<<n, ST_THREADS, 0, stream>>>(a); break;
        case 4: streams_update_kernel<T, 4, VEC><<<n, ST_THREADS, 0, stream>>>(a); break;
        case 5: streams_update_kernel<T, 5, VEC><<<n, ST_THREADS, 0, stream>>>(a); break;
        case 6: streams_update_kernel<T, 6, VEC><<<n, ST_THREADS, 0, stream>>>(a); break;
        case 7: streams_update_kernel<T, 7, VEC><<<n, ST_THREADS, 0, stream>>>(a); break;
        default: streams_update_kernel<T, 8, VEC><<<n, ST_THREADS, 0, stream>>>(a); break;
    }
}

}  // namespace liyab

using namespace liyab;

// x: float [rows of the step, S, d]; enter: float [rows, d] or null (it may not lie in x unless S is 1 and it is x); y: float
// [rows * n_sum, d] or null; ids, weights [rows * n_ids] and h [rows, d] in out_dtype with n_ids > 0; mix: float [S, S] ([from, to]), add, in: float
// [S], w: float [d], each or null; out [n, d] in out_dtype or null; rows: int [n] or null (then nothing is written to x).
extern "C" int liyab_streams_update(float* x, const float* enter, const float* y, int n_sum, const int* ids, const float* weights, int n_ids,
                                    const void* h, const float* mix, const float* add, const float* in, const float* w, float eps, void* out,
                                    int out_dtype, const int* rows, int n, int S, int d, hipStream_t stream) {
    LIYAB_REQUIRE(x && (enter || y || out), "streams_update: null pointer");
    LIYAB_REQUIRE(n >= 0 && d > 0 && S >= 1 && S <= ST_MAX_STREAMS, "streams_update: bad sizes n=%d d=%d, %d streams (up to %d)", n, d, S, ST_MAX_STREAMS);
    LIYAB_REQUIRE(y == nullptr || n_sum >= 1, "streams_update: %d rows a token", n_sum);
    LIYAB_REQUIRE(n_ids == 0 || (y && ids && weights && h && n_ids > 0 && n_ids <= n_sum), "streams_update: identity entries need the router's lists and the rows it read");
    LIYAB_REQUIRE(rows == nullptr || (y == nullptr && enter == nullptr && out), "streams_update: gathered rows are only read");
    LIYAB_REQUIRE(out_dtype == kF32 || out_dtype == kBF16, "streams_update: unknown dtype %d", out_dtype);
    if (n == 0) return 0;
    const StreamsArgs a{x, enter, y, n_sum, n_ids, ids, weights, h, mix, add, in, w, eps, out, rows, d};
    const auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    const bool vec = d % 4 == 0 && aligned(x) && aligned(enter) && aligned(y) && aligned(w) && aligned(out);
    // (thousands of rows of which a wave or less holds one: the general kernel's are shorter where nothing is left to wait for, 4,096 of 256 5.9 us against 6.2;
    // of 768 with two rows a token 9.8 against 9.1. Where rows only enter or are only read, or identity experts' rows are loaded whether one is there or not, there is
    // less to gain by loads ahead and more to run: up to some 500 rows only; us, general / this one, two streams of 768, identity experts at 300, 1,000 and 2,048 rows
    // 3.2 / 3.0, 4.3 / 4.4, 6.1 / 6.5; entering 2.8 / 2.6, 3.8 / 3.9, 5.2 / 5.7.
    // One row a token for one or two streams: up to 1,024 rows, 1,000 of two streams of 768 4.0 / 4.0, 2,048 5.7 / 6.0)
    const bool few = n_ids > 0 || y == nullptr ? n <= 512 : n_sum == 1 && S <= 2 ? n <= 1024 : n <= 2048 || d > 256;
    if (vec && d <= 4 * ST_THREADS && (y == nullptr || n_sum <= 4) && few) {
        const bool ids_in = n_ids > 0;
        const bool done = out_dtype == kF32 ? (ids_in ? launch_streams_row<float, true>(a, n, S, stream) : launch_streams_row<float, false>(a, n, S, stream))
                                            : (ids_in ? launch_streams_row<bf16_t, true>(a, n, S, stream) : launch_streams_row<bf16_t, false>(a, n, S, stream));
        if (done) return check_launch("streams_update");
    }
    if (out_dtype == kF32) {
        if (vec) launch_streams<float, 4>(a, n, S, stream);
        else launch_streams<float, 1>(a, n, S, stream);
    } else {
        if (vec) launch_streams<bf16_t, 4>(a, n, S, stream);
        else launch_streams<bf16_t, 1>(a, n, S, stream);
    }
    return check_launch("streams_update");
}
