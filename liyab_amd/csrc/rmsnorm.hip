// Root-mean-square norms over rows of the 32-bit residual stream.
//
// liyab_rmsnorm: y = x / sqrt(mean(x^2) + eps) * w, the epsilon inside the root; `rows`, when
// given, gathers (the final norm runs on the wanted rows only). Sums and the scaling are 32-bit,
// the result is rounded once to the output type.
//
// liyab_gated_norm_add: the residual update of a block whose norm stands behind its sublayer:
//   s = (y_0 + ... + y_{n_sum-1}) * sigmoid(g),   x += w * s / sqrt(mean(s^2) + eps)
// y: the sublayer's 32-bit result, one row a token or n_sum consecutive rows a token that are
// added in their order (a routed feed-forward leaves one row for each expert a token took);
// without `normalize` the sum is added as it is (x += s); with normalize = 2 the norm takes the mean off first and adds a bias,
// x += w * (s - mean(s)) / sqrt(mean((s - mean(s))^2) + eps) + b, the mean and the mean square in two passes over the row;
// g: the gate's 32-bit logits (a pointer and a row stride, so that they may be columns of a wider
// product), or none. The new row may also be written rounded to the compute type for the next
// product (`cast_out`), or, with `next_w`, what the next sublayer reads of it: the new row's own root-mean-square norm under that
// weight and `next_eps` (a block with a norm before its sublayers as well as behind them). Before a row is updated it may be kept as the request's input history of
// a causal convolution over time: `state` [slots, ring, d] holds position p at ring place p % ring,
// and the last `ring` rows of each request in the step are the ones that a later step reads.
#include "common.h"
#include "launchers.h"

namespace liyab {

template <int THREADS>
__device__ __forceinline__ float rms_block_sum(float v, float* red) {
    constexpr int WAVES = THREADS / kWave;
    v = wave_sum(v);
    if constexpr (WAVES == 1) return v;
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    __syncthreads();  // red may still be read from a previous call
    if (lane == 0) red[wave] = v;
    __syncthreads();
    float total = 0.0f;
#pragma unroll
    for (int i = 0; i < WAVES; ++i) total += red[i];
    return total;
}

template <typename T, int THREADS>
__global__ void __launch_bounds__(THREADS)
rmsnorm_kernel(T* __restrict__ out, const float* __restrict__ x, const float* __restrict__ w, const int* __restrict__ rows,
               int d, float eps) {
    __shared__ float red[THREADS / kWave];
    const int r = blockIdx.x;
    const int64_t src = rows != nullptr ? rows[r] : r;
    const float* xr = x + src * d;
    T* o = out + static_cast<int64_t>(r) * d;
    float ss = 0.0f;
    for (int i = threadIdx.x; i < d; i += THREADS) ss += xr[i] * xr[i];
    const float scale = 1.0f / sqrtf(rms_block_sum<THREADS>(ss, red) / static_cast<float>(d) + eps);
    for (int i = threadIdx.x; i < d; i += THREADS) {
        float v = xr[i] * scale;
        if (w != nullptr) v *= w[i];
        o[i] = from_float<T>(v);
    }
}

struct KeepRows {
    float* state;  // [n_slots, ring, d] or null
    int ring, n_slots;
    const int* tok_seq;
    const int* positions;
    const int* context_lens;
    const int* state_slots;
    const int* n_real;  // the number of rows that belong to a request (rows behind them are padding)
};

__device__ __forceinline__ float sigmoidf(float z) { return 1.0f / (1.0f + expf(-z)); }

// MAXV values a thread are held in registers between the two passes (d <= THREADS * MAXV); wider
// rows are read again.
template <typename T, int THREADS, int MAXV>
__global__ void __launch_bounds__(THREADS)
gated_norm_add_kernel(float* __restrict__ x, T* __restrict__ cast_out, const float* __restrict__ y, int n_sum,
                      const float* __restrict__ gate, int64_t gate_stride, const float* __restrict__ w, float eps, int normalize, int d, KeepRows keep,
                      const float* __restrict__ next_w, float next_eps, const float* __restrict__ b) {
    __shared__ float red[THREADS / kWave];
    const int t = blockIdx.x;
    float* xr = x + static_cast<int64_t>(t) * d;
    if (keep.state != nullptr && t < *keep.n_real) {
        const int s = keep.tok_seq[t], p = keep.positions[t];
        const int slot = keep.state_slots[s];
        if (p >= keep.context_lens[s] - keep.ring && slot >= 0 && slot < keep.n_slots) {
            float* dst = keep.state + (static_cast<int64_t>(slot) * keep.ring + p % keep.ring) * d;
            for (int i = threadIdx.x; i < d; i += THREADS) dst[i] = xr[i];
        }
    }
    const float* yr = y + static_cast<int64_t>(t) * n_sum * d;
    const float* gr = gate != nullptr ? gate + static_cast<int64_t>(t) * gate_stride : nullptr;
    const bool held = d <= THREADS * MAXV;
    float sv[MAXV];
    float ss = 0.0f, mean = 0.0f;
    auto value = [&](int i) {
        float s = yr[i];
        for (int k = 1; k < n_sum; ++k) s += yr[static_cast<int64_t>(k) * d + i];
        if (gr != nullptr) s *= sigmoidf(gr[i]);
        return s;
    };
    if (held) {
#pragma unroll
        for (int j = 0; j < MAXV; ++j) {
            const int i = threadIdx.x + j * THREADS;
            sv[j] = i < d ? value(i) : 0.0f;
            ss += normalize == 2 ? sv[j] : sv[j] * sv[j];
        }
    } else {
        for (int i = threadIdx.x; i < d; i += THREADS) {
            const float s = value(i);
            ss += normalize == 2 ? s : s * s;
        }
    }
    if (normalize == 2) {
        mean = rms_block_sum<THREADS>(ss, red) / static_cast<float>(d);
        ss = 0.0f;
        if (held) {
#pragma unroll
            for (int j = 0; j < MAXV; ++j) {
                sv[j] -= mean;
                if (threadIdx.x + j * THREADS < d) ss += sv[j] * sv[j];
            }
        } else {
            for (int i = threadIdx.x; i < d; i += THREADS) {
                const float s = value(i) - mean;
                ss += s * s;
            }
        }
    }
    const float scale = normalize ? 1.0f / sqrtf(rms_block_sum<THREADS>(ss, red) / static_cast<float>(d) + eps) : 1.0f;
    T* co = cast_out != nullptr ? cast_out + static_cast<int64_t>(t) * d : nullptr;
    const bool norm_next = next_w != nullptr && co != nullptr;  // what is written for the next product is the next norm of the new row
    float ss_new = 0.0f;
    auto finish = [&](int i, float s) {
        float v = s * scale;
        if (w != nullptr) v *= w[i];
        if (b != nullptr) v += b[i];
        v += xr[i];
        xr[i] = v;
        if (norm_next) ss_new += v * v;
        else if (co != nullptr) co[i] = from_float<T>(v);
        return v;
    };
    if (held) {
#pragma unroll
        for (int j = 0; j < MAXV; ++j) {
            const int i = threadIdx.x + j * THREADS;
            if (i < d) sv[j] = finish(i, sv[j]);
        }
    } else {
        for (int i = threadIdx.x; i < d; i += THREADS) finish(i, value(i) - mean);
    }
    if (norm_next) {
        const float next_scale = 1.0f / sqrtf(rms_block_sum<THREADS>(ss_new, red) / static_cast<float>(d) + next_eps);
        if (held) {
#pragma unroll
            for (int j = 0; j < MAXV; ++j) {
                const int i = threadIdx.x + j * THREADS;
                if (i < d) co[i] = from_float<T>(sv[j] * next_scale * next_w[i]);
            }
        } else {
            for (int i = threadIdx.x; i < d; i += THREADS) co[i] = from_float<T>(xr[i] * next_scale * next_w[i]);  // (each thread reads what it wrote)
        }
    }
}

// The same with a wave a row, up to 256 J values of it in registers (4 J a lane) and up to three rows of y a token: everything is asked
// for before anything is used, without a branch (a load under one is waited for where it ends), and the sums over the row need
// no barrier. A step of few rows is bound by that one trip to memory; the kernel above makes three or four in turn, and its waves
// meet at two barriers a sum (4 rows of 768 in a decode step, us: a gate 6.4 -> 4.7, with two rows a token 6.6 -> 4.4; a layer
// norm 5.4 -> 3.6, with two rows 4.0). A lane holds what lane `lane` of each of the four waves above holds, and the sums are
// added in their order: the same bits.
enum : int { kRowOnly = 0, kRowBias = 1, kRowNext = 2 };  // what else a row takes: a bias of its norm, the next norm of the new row

template <typename T, int J, int NSUM, bool GATE, int ALSO>
__global__ void __launch_bounds__(256)
gated_norm_add_wave_kernel(float* __restrict__ x, T* __restrict__ cast_out, const float* __restrict__ y, const float* __restrict__ gate, int64_t gate_stride,
                           const float* __restrict__ w, float eps, int normalize, int n, int d, KeepRows keep, const float* __restrict__ next_w,
                           float next_eps, const float* __restrict__ b) {
    constexpr int W = 4, STRIDE = W * kWave;
    const int lane = threadIdx.x % kWave, t = blockIdx.x * (blockDim.x / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    if (t >= n) return;
    float* xr = x + static_cast<int64_t>(t) * d;
    const float* yr = y + static_cast<int64_t>(t) * NSUM * d;
    const float* wp = w != nullptr ? w : xr;
    float xv[W][J], sv[W][J], yv[NSUM][W][J], gv[GATE ? W : 1][J], wv[W][J], av[ALSO ? W : 1][J];
    const auto place = [&](int q, int j) { return lane + q * kWave + j * STRIDE; };
    const auto at = [&](int q, int j) { return min(place(q, j), d - 1); };  // (past the row: its last value, counted as nothing)
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
        for (int q = 0; q < W; ++q) {
#pragma unroll
            for (int k = 0; k < NSUM; ++k) yv[k][q][j] = yr[static_cast<int64_t>(k) * d + at(q, j)];
            if constexpr (GATE) gv[q][j] = gate[static_cast<int64_t>(t) * gate_stride + at(q, j)];
        }
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
        for (int q = 0; q < W; ++q) {
            xv[q][j] = xr[at(q, j)];
            wv[q][j] = wp[at(q, j)];
            if constexpr (ALSO != kRowOnly) av[q][j] = (ALSO == kRowBias ? b : next_w)[at(q, j)];
        }
    const auto row_sum = [&](const float (&part)[W]) {
        float total = 0.0f;
#pragma unroll
        for (int q = 0; q < W; ++q) total += wave_sum(part[q]);
        return total;
    };
    float ss[W];
#pragma unroll
    for (int q = 0; q < W; ++q) {
        ss[q] = 0.0f;
#pragma unroll
        for (int j = 0; j < J; ++j) {
            float s = yv[0][q][j];
#pragma unroll
            for (int k = 1; k < NSUM; ++k) s += yv[k][q][j];
            if constexpr (GATE) s *= sigmoidf(gv[q][j]);
            sv[q][j] = place(q, j) < d ? s : 0.0f;
            ss[q] += normalize == 2 ? sv[q][j] : sv[q][j] * sv[q][j];
        }
    }
    if (normalize == 2) {
        const float mean = row_sum(ss) / static_cast<float>(d);
#pragma unroll
        for (int q = 0; q < W; ++q) {
            ss[q] = 0.0f;
#pragma unroll
            for (int j = 0; j < J; ++j) {
                sv[q][j] -= mean;
                if (place(q, j) < d) ss[q] += sv[q][j] * sv[q][j];
            }
        }
    }
    const float scale = normalize ? 1.0f / sqrtf(row_sum(ss) / static_cast<float>(d) + eps) : 1.0f;
    if (keep.state != nullptr && t < *keep.n_real) {
        const int s = keep.tok_seq[t], p = keep.positions[t];
        const int slot = keep.state_slots[s];
        if (p >= keep.context_lens[s] - keep.ring && slot >= 0 && slot < keep.n_slots) {
            float* dst = keep.state + (static_cast<int64_t>(slot) * keep.ring + p % keep.ring) * d;
#pragma unroll
            for (int j = 0; j < J; ++j)
#pragma unroll
                for (int q = 0; q < W; ++q)
                    if (place(q, j) < d) dst[place(q, j)] = xv[q][j];
        }
    }
    T* co = cast_out != nullptr ? cast_out + static_cast<int64_t>(t) * d : nullptr;
#pragma unroll
    for (int q = 0; q < W; ++q) {
        ss[q] = 0.0f;
#pragma unroll
        for (int j = 0; j < J; ++j) {
            float v = sv[q][j] * scale;
            if (w != nullptr) v *= wv[q][j];
            if constexpr (ALSO == kRowBias) v += av[q][j];
            v += xv[q][j];
            sv[q][j] = v;
            if (place(q, j) >= d) continue;
            xr[place(q, j)] = v;
            if constexpr (ALSO == kRowNext) ss[q] += v * v;
            else if (co != nullptr) co[place(q, j)] = from_float<T>(v);
        }
    }
    if constexpr (ALSO == kRowNext) {  // what is written for the next product is the next norm of the new row
        const float next_scale = 1.0f / sqrtf(row_sum(ss) / static_cast<float>(d) + next_eps);
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
            for (int q = 0; q < W; ++q)
                if (place(q, j) < d) co[place(q, j)] = from_float<T>(sv[q][j] * next_scale * av[q][j]);
    }
}

// The same with four waves a row, for up to some 1,500 rows: wave q holds what the kernel above holds as its q-th quarter, so that a row's loads, sigmoids and
// sums go side by side on four SIMDs, and the sums meet through LDS in the same order: the same bits. What a step of few rows waits for beside memory is one
// wave's sixty loads of 256 bytes and four sums in turn. us, 4 rows of 768 in a chain, before / now: 3.1 / 2.5, a layer norm
// 3.3 / 2.7, a gate 3.7 / 2.6, with two rows a token 3.8 / 2.6, the next norm too 3.5 / 2.9; 512 rows 3.4 / 2.9, a gate 4.1 / 3.1.
template <typename T, int J, int NSUM, bool GATE, int ALSO>
__global__ void __launch_bounds__(256)
gated_norm_add_quarters_kernel(float* __restrict__ x, T* __restrict__ cast_out, const float* __restrict__ y, const float* __restrict__ gate, int64_t gate_stride,
                               const float* __restrict__ w, float eps, int normalize, int n, int d, KeepRows keep, const float* __restrict__ next_w,
                               float next_eps, const float* __restrict__ b) {
    constexpr int W = 4, STRIDE = W * kWave;
    __shared__ float meet[3][W];  // the quarters' sums: the mean's, the mean square's, the next norm's
    const int lane = threadIdx.x % kWave, q = threadIdx.x / kWave, t = blockIdx.x;
    float* xr = x + static_cast<int64_t>(t) * d;
    const float* yr = y + static_cast<int64_t>(t) * NSUM * d;
    const float* wp = w != nullptr ? w : xr;
    float xv[J], sv[J], yv[NSUM][J], gv[J], wv[J], av[J];
    const auto place = [&](int j) { return static_cast<int>(threadIdx.x) + j * STRIDE; };
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int at = min(place(j), d - 1);  // (past the row: its last value, counted as nothing)
#pragma unroll
        for (int k = 0; k < NSUM; ++k) yv[k][j] = yr[static_cast<int64_t>(k) * d + at];
        if constexpr (GATE) gv[j] = gate[static_cast<int64_t>(t) * gate_stride + at];
        xv[j] = xr[at];
        wv[j] = wp[at];
        if constexpr (ALSO != kRowOnly) av[j] = (ALSO == kRowBias ? b : next_w)[at];
    }
    // where the old row is kept: looked up while the row is on its way
    float* kept = nullptr;
    if (keep.state != nullptr && t < *keep.n_real) {
        const int s = keep.tok_seq[t], p = keep.positions[t];
        const int slot = keep.state_slots[s];
        if (p >= keep.context_lens[s] - keep.ring && slot >= 0 && slot < keep.n_slots) kept = keep.state + (static_cast<int64_t>(slot) * keep.ring + p % keep.ring) * d;
    }
    const auto row_sum = [&](float part, int which) {
        part = wave_sum(part);
        if (lane == 0) meet[which][q] = part;
        lds_barrier();
        float total = 0.0f;
#pragma unroll
        for (int i = 0; i < W; ++i) total += meet[which][i];
        return total;
    };
    float ss = 0.0f;
#pragma unroll
    for (int j = 0; j < J; ++j) {
        float s = yv[0][j];
#pragma unroll
        for (int k = 1; k < NSUM; ++k) s += yv[k][j];
        if constexpr (GATE) s *= sigmoidf(gv[j]);
        sv[j] = place(j) < d ? s : 0.0f;
        ss += normalize == 2 ? sv[j] : sv[j] * sv[j];
    }
    if (normalize == 2) {
        const float mean = row_sum(ss, 0) / static_cast<float>(d);
        ss = 0.0f;
#pragma unroll
        for (int j = 0; j < J; ++j) {
            sv[j] -= mean;
            if (place(j) < d) ss += sv[j] * sv[j];
        }
    }
    const float scale = normalize ? 1.0f / sqrtf(row_sum(ss, 1) / static_cast<float>(d) + eps) : 1.0f;
    T* co = cast_out != nullptr ? cast_out + static_cast<int64_t>(t) * d : nullptr;
    ss = 0.0f;
#pragma unroll
    for (int j = 0; j < J; ++j) {
        float v = sv[j] * scale;
        if (w != nullptr) v *= wv[j];
        if constexpr (ALSO == kRowBias) v += av[j];
        v += xv[j];
        sv[j] = v;
        if (place(j) >= d) continue;
        if (kept != nullptr) kept[place(j)] = xv[j];
        xr[place(j)] = v;
        if constexpr (ALSO == kRowNext) ss += v * v;
        else if (co != nullptr) co[place(j)] = from_float<T>(v);
    }
    if constexpr (ALSO == kRowNext) {  // what is written for the next product is the next norm of the new row
        const float next_scale = 1.0f / sqrtf(row_sum(ss, 2) / static_cast<float>(d) + next_eps);
#pragma unroll
        for (int j = 0; j < J; ++j)
            if (place(j) < d) co[place(j)] = from_float<T>(sv[j] * next_scale * av[j]);
    }
}

// Whether the wave kernel took the rows (of the gate, a bias and the next norm it takes one: what the blocks that exist use); if
// not, the one above does. A place past the row costs what one inside does, which shows where each takes a sigmoid: with a gate J is
// the least that holds the row (behind the kernels that write y and the gate, us for all of them, by workgroups, by waves with J of 3, 4
// and 8 only, and now: 4 rows of 256 6.0, 6.3, 5.6; of 1,280 8.2, 9.3, 8.4; 2,048 rows of 1,280 21.1, 21.7, 19.3. Bokulix 1,280 wide, a
// prompt of 32 and eight decoded tokens, 29.8, 29.1, 28.1 ms). Without one, J of 3, 4 and 8 is enough (behind the kernel that writes y, by
// workgroups and by waves: 4 rows of 1,280 5.4 and 5.4, with two rows a token 6.7 and 5.7; 2,048 rows of 1,280 13.7 and 12.9; of 2,048 18.6 and
// 16.6, a layer norm 21.2 and 16.9, three rows a token and the next norm 33.6 and 30.8).
// Rows up to which four waves share one: while they do not fill the chip (512 rows of 320 to 2,048 0.73 with a gate and 0.79 to 0.80 of a wave a row, 1,500 0.82
// and 0.86 to 0.88; 2,048 rows of 320 1.03 and 1.00, of 2,048 0.84 and 0.92; 4,096 even).
constexpr int kQuarterRows = 1536;
template <typename T>
bool gated_norm_add_by_waves(float* x, T* cast_out, const float* y, int n_sum, const float* gate, int64_t gate_stride, const float* w, float eps, int normalize,
                             int n, int d, const KeepRows& keep, const float* next_w, float next_eps, const float* b, hipStream_t stream) {
    if (d > 2048 || n_sum > 3 || (gate != nullptr) + (b != nullptr) + (next_w != nullptr) > 1) return false;
#define LIYAB_ROWS(KERNEL, THREADS, ROWS, J, S, G, A) \
    KERNEL<T, J, S, G, A><<<(n + ROWS - 1) / ROWS, THREADS, 0, stream>>>(x, cast_out, y, gate, gate_stride, w, eps, normalize, n, d, keep, next_w, next_eps, b)
#define LIYAB_GO(J, S, G, A)                                                                            \
    do {                                                                                                \
        if (n <= kQuarterRows) LIYAB_ROWS(gated_norm_add_quarters_kernel, 4 * kWave, 1, J, S, G, A);    \
        else LIYAB_ROWS(gated_norm_add_wave_kernel, 4 * kWave, 4, J, S, G, A);                          \
    } while (0)
#define LIYAB_SUMS(J, G, A)                 \
    do {                                    \
        if (n_sum == 1) LIYAB_GO(J, 1, G, A); \
        else if (n_sum == 2) LIYAB_GO(J, 2, G, A); \
        else LIYAB_GO(J, 3, G, A);          \
    } while (0)
#define LIYAB_WIDTHS(A)                         \
    do {                                        \
        if (d <= 768) LIYAB_SUMS(3, false, A);  \
        else if (d <= 1024) LIYAB_SUMS(4, false, A); \
        else LIYAB_SUMS(8, false, A);           \
    } while (0)
    if (gate != nullptr) {
        switch ((d + 255) / 256) {
            case 1: LIYAB_SUMS(1, true, kRowOnly); break;
            case 2: LIYAB_SUMS(2, true, kRowOnly); break;
            case 3: LIYAB_SUMS(3, true, kRowOnly); break;
            case 4: LIYAB_SUMS(4, true, kRowOnly); break;
            case 5: LIYAB_SUMS(5, true, kRowOnly); break;
            case 6: LIYAB_SUMS(6, true, kRowOnly); break;
            case 7: LIYAB_SUMS(7, true, kRowOnly); break;
            default: LIYAB_SUMS(8, true, kRowOnly); break;
        }
    } else if (b != nullptr) {
        LIYAB_WIDTHS(kRowBias);
    } else if (next_w != nullptr) {
        LIYAB_WIDTHS(kRowNext);
    } else {
        LIYAB_WIDTHS(kRowOnly);
    }
#undef LIYAB_ROWS
#undef LIYAB_WIDTHS
#undef LIYAB_SUMS
#undef LIYAB_GO
    return true;
}

}  // namespace liyab

using namespace liyab;

extern "C" int liyab_rmsnorm(void* out, int out_dtype, const float* x, const float* w, const int* rows, int n, int d, float eps,
                             hipStream_t stream) {
    LIYAB_REQUIRE(out && x, "rmsnorm: null pointer");
    LIYAB_REQUIRE(n >= 0 && d > 0, "rmsnorm: bad sizes n=%d d=%d", n, d);
    LIYAB_REQUIRE(out_dtype == kF32 || out_dtype == kBF16, "rmsnorm: unknown dtype %d", out_dtype);
    if (n == 0) return 0;
    if (out_dtype == kF32)
        rmsnorm_kernel<float, 256><<<n, 256, 0, stream>>>(static_cast<float*>(out), x, w, rows, d, eps);
    else
        rmsnorm_kernel<bf16_t, 256><<<n, 256, 0, stream>>>(static_cast<bf16_t*>(out), x, w, rows, d, eps);
    return check_launch("rmsnorm");
}

extern "C" int liyab_gated_norm_add(float* x, void* cast_out, int cast_dtype, const float* y, int n_sum, const float* gate,
                                    int64_t gate_stride, const float* w, float eps, int normalize, int n, int d, float* state, int ring, int n_slots,
                                    const int* tok_seq, const int* positions, const int* context_lens, const int* state_slots,
                                    const int* n_real, const float* next_w, float next_eps, const float* b, hipStream_t stream) {
    LIYAB_REQUIRE(x && y, "gated_norm_add: null pointer");
    LIYAB_REQUIRE(normalize >= 0 && normalize <= 2, "gated_norm_add: unknown norm %d", normalize);
    LIYAB_REQUIRE(next_w == nullptr || cast_out != nullptr, "gated_norm_add: the next norm's rows need a place");
    LIYAB_REQUIRE(n >= 0 && d > 0 && n_sum >= 1, "gated_norm_add: bad sizes n=%d d=%d n_sum=%d", n, d, n_sum);
    LIYAB_REQUIRE(cast_dtype == kF32 || cast_dtype == kBF16, "gated_norm_add: unknown dtype %d", cast_dtype);
    LIYAB_REQUIRE(gate == nullptr || gate_stride >= d, "gated_norm_add: the gate's row stride is shorter than a row");
    LIYAB_REQUIRE(state == nullptr || (ring > 0 && n_slots > 0 && tok_seq && positions && context_lens && state_slots && n_real),
                  "gated_norm_add: rows are kept only with a ring, slots and the step's tables");
    if (n == 0) return 0;
    const KeepRows keep{state, ring, n_slots, tok_seq, positions, context_lens, state_slots, n_real};
    if (cast_dtype == kF32 ? gated_norm_add_by_waves(x, static_cast<float*>(cast_out), y, n_sum, gate, gate_stride, w, eps, normalize, n, d, keep, next_w, next_eps, b, stream)
                           : gated_norm_add_by_waves(x, static_cast<bf16_t*>(cast_out), y, n_sum, gate, gate_stride, w, eps, normalize, n, d, keep, next_w, next_eps, b, stream))
        return check_launch("gated_norm_add");
    if (cast_dtype == kF32)
        gated_norm_add_kernel<float, 256, 8><<<n, 256, 0, stream>>>(x, static_cast<float*>(cast_out), y, n_sum, gate, gate_stride, w, eps, normalize, d, keep, next_w, next_eps, b);
    else
        gated_norm_add_kernel<bf16_t, 256, 8><<<n, 256, 0, stream>>>(x, static_cast<bf16_t*>(cast_out), y, n_sum, gate, gate_stride, w, eps, normalize, d, keep, next_w, next_eps, b);
    return check_launch("gated_norm_add");
}
