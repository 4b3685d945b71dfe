// out[M,N] = a[M,K] . w[N,K]^T in bfloat16 for steps of few tokens in the batch-invariant mode: the bits of
// gemm_mfma_dl.hip's tiles of four sums (unit u of 64 k goes to sum u % 4, 16 k an instruction of 32 x 32, the
// sums added in their order), from kernels that stream the weights and make the first operand themselves.
//
// A workgroup owns NB output features and up to 32 rows, and each of its four waves walks one of the four sums. The first operand is
//   rows     bfloat16 rows: both operands go through a ring in LDS of the wave's own (no barrier: a wave waits for its own loads), 8 rows of
//            64 k a load, up to twelve units in flight;
//   norm     LayerNorm of 32-bit rows, computed by every workgroup while its weights are on their way, with
//            layernorm.hip's operations: the same bits as the norm's own kernel, without its link in the step's chain;
//   splits   attention's splits, merged with attention_merge_kernel's operations: again the same bits without its link.
// For the latter two the rows go to LDS in bfloat16 and the weights straight into registers (three units, or six, in flight: a wait for a row
// asked for ahead of them is no wait for them, which it is for the compiler where they go to LDS). With fewer than 32 features or rows the
// matrix operands' other lanes repeat some; their results are dropped.
#include "common.h"
#include "launchers.h"
#include "epilogue.h"
#include "ring.h"

namespace liyab {
namespace by_rows {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(16))) float floatx16;
typedef __attribute__((ext_vector_type(4))) float floatx4;
typedef __attribute__((ext_vector_type(2))) float floatx2;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

union Frag {
    u32x4 u;
    bf16x8 v;
};

enum : int { kRows = 0, kNorm = 1, kSplits = 2 };
constexpr int SUMS = 4, ROWS = 32, UNIT = 64;  // sums, and waves; rows a workgroup; k of a unit

struct Source {
    const bf16_t* a;  // rows: [M, lda]
    int64_t lda;
    const float* x;  // norm: [M, K]; splits: [M][n_head][n_splits][hd + 4]
    const float* weight;
    const float* bias;
    float eps;
    int n_splits, n_head, hd;
};

// A workgroup's LDS: the waves' rings (whose place the sums take at the end), and behind them rows made here.
template <int NB, int MR, int RING>
constexpr size_t ring_bytes() {
    constexpr size_t ring = MR > 0 ? static_cast<size_t>(SUMS) * RING * (NB + MR) * UNIT * 2 : 0, sums = static_cast<size_t>(SUMS) * NB * (ROWS + 1) * 4;
    return ring > sums ? ring : sums;
}

// MR: rows of the ring (rows: 8, 16 or 32, M rounded up; otherwise 0). RING: units of the ring, or (norm, splits) sets of three units in
// registers, 1 or 2. FORM: pieces of 4 a lane of a row (norm), splits merged at most (splits), not read (rows).
// EPI: the epilogue, fixed at compile time (the rarer activations: -1): a kernel this short waits for its own instructions, cold in every launch of a chain
// (norm and product at 768 -> 3,072, 8 rows: 4.6 us with all epilogues and three forms of the norm in 3,300 instructions, 4.2 with 1,400).
template <typename OutT, int NB, int MR, int SRC, int FORM, int RING, int EPI>
__global__ void __launch_bounds__(64 * SUMS)
gemm_rows_kernel(Source src, const bf16_t* __restrict__ w, int M_all, int N, int K, EpiParams epi) {
    static_assert((SRC == kRows) == (MR > 0) && NB % 8 == 0 && MR % 8 == 0, "whole loads");
    constexpr int W_LOADS = NB / 8, A_LOADS = MR / 8, LOADS = W_LOADS + A_LOADS, SLOT = (NB + MR) * UNIT;  // a load: 8 rows of 64 k
    static_assert((RING - 1) * LOADS <= 63, "the counter of loads in flight has six bits");
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    float* const red = reinterpret_cast<float*>(smem);  // [sum][NB][ROWS + 1]
    bf16_t* const xs = reinterpret_cast<bf16_t*>(smem + ring_bytes<NB, MR, RING>());  // [M][K + 8]
    const int ldx = K + 8;  // rows 16 bytes apart modulo the banks
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int li = lane % 32, g = lane / 32;
    const int row0 = blockIdx.y * ROWS, M = min(ROWS, M_all - row0), n0 = blockIdx.x * NB;
    const int units = K / UNIT, mine = (units - wave + SUMS - 1) / SUMS;  // this wave's units: wave, wave + 4, ...
    bf16_t* const ring = reinterpret_cast<bf16_t*>(smem) + wave * RING * SLOT;

    // this lane's part in a load: row lane / 8 of the 8, piece lane % 8
    const int lrow = lane / 8, lpos = lane % 8;
    const bf16_t* from[LOADS];
#pragma unroll
    for (int i = 0; i < W_LOADS; ++i) from[i] = w + static_cast<int64_t>(min(n0 + 8 * i + lrow, N - 1)) * K + (lpos ^ ring_swizzle(8 * i + lrow)) * 8;
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i)
        from[W_LOADS + i] = src.a + static_cast<int64_t>(row0 + min(8 * i + lrow, M - 1)) * src.lda + (lpos ^ ring_swizzle(8 * i + lrow)) * 8;
    // unit i of this wave's into place `slot` (one past the end of K: the last one again, not multiplied)
    auto load = [&](int i, int slot) {
        const int k = min(wave + SUMS * i, units - 1) * UNIT;
#pragma unroll
        for (int l = 0; l < LOADS; ++l) {
            const bf16_t* const piece = from[l] + k;
            bf16_t* const to = ring + slot * SLOT + l * 8 * UNIT;
            __builtin_amdgcn_global_load_lds(piece, (lds_void_ptr)to, 16, 0, 0);
        }
    };
    // the same three units at a time into registers, as the matrix core takes them
    constexpr int SET = 3;
    Frag fw[SRC == kRows ? 1 : RING][SET][4];
    const bf16_t* const wlane = w + static_cast<int64_t>(min(n0 + li % NB, N - 1)) * K + g * 8;
    auto load_set = [&](int i0, int set) {
#pragma unroll
        for (int t = 0; t < SET; ++t)
#pragma unroll
            for (int s = 0; s < 4; ++s)
                fw[set][t][s].u = *reinterpret_cast<const u32x4*>(wlane + min(wave + SUMS * (i0 + t), units - 1) * UNIT + 16 * s);
    };

    // This thread's first output and what its epilogue reads, its bias and one word more: the row's slot or the value it is added to. No
    // load under a branch, which would be waited for where the branch ends: who has nothing to read gets a word of the weights.
    const int e_m = row0 + min(tid / NB, M - 1), e_n = min(n0 + tid % NB, N - 1);
    typedef const __attribute__((address_space(1))) float* global_floats;
    const auto nothing = (global_floats)(w);
    auto bias_at = epi.bias != nullptr ? (global_floats)(epi.bias + e_n) : nothing;
    auto word_at = EPI == kEpiResidual   ? (global_floats)(epi.residual + static_cast<int64_t>(e_m) * epi.ldr + e_n)
                   : EPI == kEpiQkvPaged ? (global_floats)(epi.slots + e_m)
                                              : nothing;
    asm volatile("" : "+v"(bias_at), "+v"(word_at));  // (worked out here, ahead of every load)
    float e_bias;
    float e_word;
    auto ask = [&]() {
        if constexpr (SRC == kRows) {
            e_bias = *bias_at;
            e_word = *word_at;
            // (no load may cross to the other side: the waits below count on what is asked for behind them)
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int p = 0; p < RING; ++p) load(p, p);
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("" ::: "memory");
        } else {
#pragma unroll
            for (int p = 0; p < RING; ++p) load_set(SET * p, p);
            e_bias = *bias_at;
            e_word = *word_at;
        }
    };

    if constexpr (SRC == kRows) {
        ask();
    } else if constexpr (SRC == kNorm) {
        // a wave's rows two at a time, each in registers; the row's loads go ahead of the weights': a wait for the row is then
        // no wait for the weights
        const int nv = K / 4;
        const floatx4 zero = {0.0f, 0.0f, 0.0f, 0.0f}, one = {1.0f, 1.0f, 1.0f, 1.0f};
        const float* const weight = src.weight != nullptr ? src.weight : src.x;  // (without one: a row's values, read and dropped)
        const float* const bias = src.bias != nullptr ? src.bias : src.x;
        auto norm_rows = [&](int m, auto&& between) {  // rows m and m + 4 (past the last: the last again, not kept)
            constexpr int R = 2;
            floatx4 v[R][FORM], gw[FORM], gb[FORM];
#pragma unroll
            for (int j = 0; j < FORM; ++j) {
                const int at = min(lane + kWave * j, nv - 1);  // past the row: its last piece again, unused
#pragma unroll
                for (int r = 0; r < R; ++r) v[r][j] = reinterpret_cast<const floatx4*>(src.x + static_cast<int64_t>(row0 + min(m + SUMS * r, M - 1)) * K)[at];
                gw[j] = reinterpret_cast<const floatx4*>(weight)[at];
                gb[j] = reinterpret_cast<const floatx4*>(bias)[at];
            }
            between();
            __builtin_amdgcn_sched_barrier(0);  // keep the loads in this order: the scheduler would sink them to their use
            float mean[R], scale[R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                float s = 0.0f;
#pragma unroll
                for (int j = 0; j < FORM; ++j)
                    if (lane + kWave * j < nv) s += (v[r][j][0] + v[r][j][1]) + (v[r][j][2] + v[r][j][3]);
                mean[r] = wave_sum(s) / static_cast<float>(K);
            }
#pragma unroll
            for (int r = 0; r < R; ++r) {
                float ss = 0.0f;
#pragma unroll
                for (int j = 0; j < FORM; ++j)
                    if (lane + kWave * j < nv) {
                        const floatx4 dev = v[r][j] - mean[r];
                        ss += (dev[0] * dev[0] + dev[1] * dev[1]) + (dev[2] * dev[2] + dev[3] * dev[3]);
                    }
                scale[r] = 1.0f / sqrtf(wave_sum(ss) / static_cast<float>(K) + src.eps);
            }
#pragma unroll
            for (int j = 0; j < FORM; ++j) {
                gw[j] = src.weight != nullptr ? gw[j] : one;
                gb[j] = src.bias != nullptr ? gb[j] : zero;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const floatx4 y = (v[r][j] - mean[r]) * scale[r] * gw[j] + gb[j];
                    const float four[4] = {y[0], y[1], y[2], y[3]};
                    if (lane + kWave * j < nv && m + SUMS * r < M) store4<bf16_t>(xs + (m + SUMS * r) * ldx + 4 * (lane + kWave * j), four);
                }
            }
        };
        if (wave < M) norm_rows(wave, ask);
        else ask();
        for (int m = wave + 2 * SUMS; m < M; m += 2 * SUMS) norm_rows(m, []() {});
        lds_barrier();  // the weights may still be on their way
    } else {
        // four consecutive k of a token a thread and item, merged over the splits; ITEMS items' loads in flight together
        constexpr int ITEMS = FORM <= 4 ? 3 : 2;
        const int S = src.n_splits, hd4 = src.hd + 4, per = K / 4, items = M * per;
        struct Item {
            floatx4 acc[FORM];
            floatx2 ml[FORM];
            int place;
        } it[ITEMS];
        auto fetch = [&](int first) {
#pragma unroll
            for (int i = 0; i < ITEMS; ++i) {
                const int n = first + i * 64 * SUMS, nc = min(n, items - 1);  // past the end: the last one again, dropped
                const int m = nc / per, k = (nc - m * per) * 4, head = k / src.hd;
                const float* p = src.x + (static_cast<int64_t>(row0 + m) * src.n_head + head) * S * hd4;
                it[i].place = n < items ? m * ldx + k : -1;
#pragma unroll
                for (int s = 0; s < FORM; ++s) it[i].ml[s] = *reinterpret_cast<const floatx2*>(p + min(s, S - 1) * hd4 + src.hd);
#pragma unroll
                for (int s = 0; s < FORM; ++s) it[i].acc[s] = *reinterpret_cast<const floatx4*>(p + min(s, S - 1) * hd4 + k - head * src.hd);
            }
        };
        auto finish = [&]() {
#pragma unroll
            for (int i = 0; i < ITEMS; ++i) {
                float mx = -INFINITY;
#pragma unroll
                for (int s = 0; s < FORM; ++s)
                    if (s < S) mx = fmaxf(mx, it[i].ml[s][0]);
                float sum = 0.0f, o[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int s = 0; s < FORM; ++s) {
                    if (s >= S || it[i].ml[s][0] == -INFINITY) continue;
                    const float f = __expf(it[i].ml[s][0] - mx);
                    sum = fmaf(f, it[i].ml[s][1], sum);
#pragma unroll
                    for (int c = 0; c < 4; ++c) o[c] = fmaf(f, it[i].acc[s][c], o[c]);
                }
                const float four[4] = {o[0] / sum, o[1] / sum, o[2] / sum, o[3] / sum};
                if (it[i].place >= 0) store4<bf16_t>(xs + it[i].place, four);
            }
        };
        fetch(tid);
        ask();
        __builtin_amdgcn_sched_barrier(0);
        finish();
        for (int n = tid + ITEMS * 64 * SUMS; n < items; n += ITEMS * 64 * SUMS) {
            fetch(n);
            finish();
        }
        lds_barrier();
    }

    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
    if constexpr (SRC == kRows) {
        const int wrow = li % NB, arow = min(li, M - 1);
        auto multiply = [&](int slot) {
            const bf16_t* const sw = ring + slot * SLOT + wrow * UNIT;
            const bf16_t* const sa = ring + slot * SLOT + (NB + arow) * UNIT;
            Frag x[4], y[4];
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                x[s].u = *reinterpret_cast<const u32x4*>(sw + ((2 * s + g) ^ ring_swizzle(wrow)) * 8);
                y[s].u = *reinterpret_cast<const u32x4*>(sa + ((2 * s + g) ^ ring_swizzle(arow)) * 8);
            }
#pragma unroll
            for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[s].v, y[s].v, acc, 0, 0, 0);
        };
        // unit after unit: the later ones of the ring may still be on their way (a wave's loads complete in order)
        int i0 = 0;
        for (; i0 + RING < mine; i0 += RING) {
#pragma unroll
            for (int t = 0; t < RING; ++t) {
                wait_loads<(RING - 1) * LOADS>();
                multiply(t);
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the place has been read
                load(i0 + RING + t, t);
            }
        }
        in_turn(std::make_integer_sequence<int, RING>{}, [&](auto at) {
            constexpr int t = decltype(at)::value;
            wait_loads<(RING - 1 - t) * LOADS>();
            if (i0 + t < mine) multiply(t);
        });
        lds_barrier();  // (the sums take the rings' place)
    } else {
        const bf16_t* const xrow = xs + min(li, M - 1) * ldx + g * 8;
        auto multiply = [&](int i0, int set) {
#pragma unroll
            for (int t = 0; t < SET; ++t) {
                if (i0 + t >= mine) break;
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    Frag x;
                    x.u = *reinterpret_cast<const u32x4*>(xrow + (wave + SUMS * (i0 + t)) * UNIT + 16 * s);
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fw[set][t][s].v, x.v, acc, 0, 0, 0);
                }
            }
        };
        int i0 = 0;
        if constexpr (RING == 2) {
            for (; i0 + 2 * SET < mine; i0 += 2 * SET) {
                multiply(i0, 0);
                load_set(i0 + 2 * SET, 0);
                __builtin_amdgcn_sched_barrier(0);
                multiply(i0 + SET, 1);
                load_set(i0 + 3 * SET, 1);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        multiply(i0, 0);
        if constexpr (RING == 2) multiply(i0 + SET, 1);
    }

    // acc[r] = this sum of feature 8 (r / 4) + 4 g + r % 4 and row li
#pragma unroll
    for (int r = 0; r < NB / 2; ++r) red[(wave * NB + 8 * (r / 4) + 4 * g + r % 4) * (ROWS + 1) + li] = acc[r];
    lds_barrier();
    for (int e = tid; e < M * NB; e += 64 * SUMS) {
        const int m = e / NB, j = e % NB, n = n0 + j;
        if (n >= N) continue;
        float v = red[j * (ROWS + 1) + m];
#pragma unroll
        for (int q = 1; q < SUMS; ++q) v += red[(q * NB + j) * (ROWS + 1) + m];
        // (a thread's later outputs read what they need here)
        const bool first = e == tid;
        const float bias = first ? e_bias : epi.bias != nullptr ? epi.bias[n] : 0.0f;
        if (epi.bias != nullptr) v += bias;
        if constexpr (EPI == kEpiResidual) {
            float* const at = epi.residual + static_cast<int64_t>(row0 + m) * epi.ldr + n;
            *at = (first ? e_word : *at) + v;
        } else if constexpr (EPI == kEpiQkvPaged) {
            if (n < epi.q_dim) {
                static_cast<OutT*>(epi.out)[static_cast<int64_t>(row0 + m) * epi.ldo + n] = from_float<OutT>(v);
            } else {
                const int64_t at = qkv_row_base(epi, first ? __float_as_int(e_word) : epi.slots[row0 + m]);
                if (at < 0) continue;
                const bool is_v = n >= epi.q_dim + epi.kv_dim;
                const int c = n - epi.q_dim - (is_v ? epi.kv_dim : 0), head = c / epi.hd;
                static_cast<OutT*>(is_v ? epi.vc : epi.kc)[at + static_cast<int64_t>(head) * epi.page_size * epi.hd + (c - head * epi.hd)] = from_float<OutT>(v);
            }
        } else {
            epilogue_store_biased<OutT, EPI>(epi, row0 + m, n, v);
        }
    }
}

template <typename OutT, int NB, int MR, int SRC, int FORM, int RING, int EPI>
int launch_as(const Source& src, const bf16_t* w, int M, int N, int K, const EpiParams& epi, hipStream_t stream) {
    const size_t smem = ring_bytes<NB, MR, RING>() + (SRC == kRows ? 0 : static_cast<size_t>(M < ROWS ? M : ROWS) * (K + 8) * 2);
    LIYAB_REQUIRE(smem <= 160 * 1024, "gemm_rows: %d rows of %d need %zu bytes of LDS", M, K, smem);
    auto kern = gemm_rows_kernel<OutT, NB, MR, SRC, FORM, RING, EPI>;
    static bool ready = false;  // once per instantiation, outside any stream capture's first use
    if (!ready) {
        hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        ready = true;
    }
    kern<<<dim3((N + NB - 1) / NB, (M + ROWS - 1) / ROWS), 64 * SUMS, smem, stream>>>(src, w, M, N, K, epi);
    return check_launch("gemm_rows");
}

// The units a wave has in flight: all of them up to 768 k; beyond, as many as the LDS holds of 6 and 12, or six in registers.
template <typename OutT, int NB, int MR, int SRC, int FORM, int EPI>
int launch_ring(const Source& src, const bf16_t* w, int M, int N, int K, const EpiParams& epi, hipStream_t stream) {
    const int units = (K / UNIT + SUMS - 1) / SUMS;  // a wave's
    if constexpr (SRC == kRows) {
        constexpr int most = 288 / (NB + MR);
        if constexpr (most >= 12)
            if (units > 6) return launch_as<OutT, NB, MR, SRC, FORM, 12, EPI>(src, w, M, N, K, epi, stream);
        if constexpr (most >= 6)
            if (units > 3) return launch_as<OutT, NB, MR, SRC, FORM, 6, EPI>(src, w, M, N, K, epi, stream);
        return launch_as<OutT, NB, MR, SRC, FORM, 3, EPI>(src, w, M, N, K, epi, stream);
    } else {
        return units > 3 ? launch_as<OutT, NB, MR, SRC, FORM, 2, EPI>(src, w, M, N, K, epi, stream) : launch_as<OutT, NB, MR, SRC, FORM, 1, EPI>(src, w, M, N, K, epi, stream);
    }
}
template <typename OutT, int NB, int SRC, int EPI>
int launch_form(const Source& src, const bf16_t* w, int M, int N, int K, const EpiParams& epi, hipStream_t stream) {
    if constexpr (SRC == kRows) {
        if (M <= 8) return launch_ring<OutT, NB, 8, SRC, 0, EPI>(src, w, M, N, K, epi, stream);
        if (M <= 16) return launch_ring<OutT, NB, 16, SRC, 0, EPI>(src, w, M, N, K, epi, stream);
        return launch_ring<OutT, NB, 32, SRC, 0, EPI>(src, w, M, N, K, epi, stream);
    } else if constexpr (SRC == kNorm) {
        if (K <= 768) return launch_ring<OutT, NB, 0, SRC, 3, EPI>(src, w, M, N, K, epi, stream);
        return K <= 1024 ? launch_ring<OutT, NB, 0, SRC, 4, EPI>(src, w, M, N, K, epi, stream) : launch_ring<OutT, NB, 0, SRC, 8, EPI>(src, w, M, N, K, epi, stream);
    } else {
        return src.n_splits <= 4 ? launch_ring<OutT, NB, 0, SRC, 4, EPI>(src, w, M, N, K, epi, stream) : launch_ring<OutT, NB, 0, SRC, 8, EPI>(src, w, M, N, K, epi, stream);
    }
}

template <typename OutT, int SRC, int EPI>
int launch_strip(const Source& src, const bf16_t* w, int M, int N, int K, int strip, const EpiParams& epi, hipStream_t stream) {
    if (strip == 0) {
        // the narrowest strips that still have a compute unit each (128 combinations of K and N up to 8,192, 1 to 64 rows: within 3 % of the best of the
        // three on average); a vocabulary's worth of features in strips of 16 while K is short (8 rows, 768 -> 50,257: 15.3 us against 15.7 in strips
        // of 32, 1,024 -> 50,257 23.7 against 25.7; 1,600 -> 16,384 19.2 against 12.2), past 768 k only up to 8 rows: with the rings of 16 rows or more a workgroup
        // of 16 features fills a compute unit (16 rows, 1,024 -> 50,257 37.1 against 30.8, 1,280 -> 16,384 15.2 against 12.2; 768 -> 50,257 17.5 against 18.5). A norm is repeated by every workgroup: wider ones
        // there (1,024 -> 4,096, 8 rows: 6.1 us in strips of 32, 6.4 in strips of 16)
        const int tiles = (M + ROWS - 1) / ROWS, most = SRC == kNorm ? 192 : 256;
        strip = SRC != kNorm && (N + 7) / 8 * tiles <= most ? 8 : (N + 15) / 16 * tiles <= most ? 16 : 32;
        if (SRC == kRows && N > 32 * 256 && K <= (M <= 8 ? 1280 : 768)) strip = 16;
    }
    switch (strip) {
        case 8: return launch_form<OutT, 8, SRC, EPI>(src, w, M, N, K, epi, stream);
        case 16: return launch_form<OutT, 16, SRC, EPI>(src, w, M, N, K, epi, stream);
        case 32: return launch_form<OutT, 32, SRC, EPI>(src, w, M, N, K, epi, stream);
        default: return fail(1, "gemm_rows: strips of %d features (8, 16 or 32)", strip);
    }
}

template <int SRC>
int launch_epi(const Source& src, const bf16_t* w, int M, int N, int K, int strip, const EpiParams& epi, hipStream_t stream) {
#define LIYAB_ROWS(OUT, EPI) launch_strip<OUT, SRC, EPI>(src, w, M, N, K, strip, epi, stream)
    if constexpr (SRC != kNorm)
        if (epi.mode == kEpiResidual) return LIYAB_ROWS(float, kEpiResidual);
    if constexpr (SRC != kSplits) {
        if (epi.out_dtype == kF32) {
            LIYAB_REQUIRE(epi.mode != kEpiQkvPaged, "gemm_rows: bfloat16 rows go to bfloat16 pages");
            if (SRC == kRows && epi.mode == kEpiNone) return LIYAB_ROWS(float, kEpiNone);
            if (epi.mode <= kEpiGeluErf) return LIYAB_ROWS(float, -1);
        } else {
            if (epi.mode == kEpiGeluTanh) return LIYAB_ROWS(bf16_t, kEpiGeluTanh);
            if (epi.mode == kEpiQkvPaged) return LIYAB_ROWS(bf16_t, kEpiQkvPaged);
            if (epi.mode <= kEpiGeluErf) return LIYAB_ROWS(bf16_t, -1);
        }
    }
#undef LIYAB_ROWS
    return fail(1, "gemm_rows: epilogue %d is not taken", epi.mode);
}

static bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }
static int check_rows(const void* w, int M, int N, int K, const EpiParams* epi) {
    LIYAB_REQUIRE(w && epi, "gemm_rows: null operand");
    LIYAB_REQUIRE(M >= 0 && M <= 64 && N > 0 && K > 0 && K % 64 == 0, "gemm_rows: bad sizes M=%d (at most 64) N=%d K=%d (a multiple of 64)", M, N, K);
    LIYAB_REQUIRE(al16(w), "gemm_rows: operands must be 16-byte aligned");
    return check_epilogue(*epi, M, N);
}

}  // namespace by_rows
}  // namespace liyab

using namespace liyab;
using namespace liyab::by_rows;

// M <= 64 rows, K a multiple of 64, w [N, K] bfloat16; strip: output features a workgroup, 8, 16 or 32 (0: chosen from N).
extern "C" int liyab_gemm_rows(const void* a, int64_t lda, const void* w, int M, int N, int K, int strip, const EpiParams* epi, hipStream_t stream) {
    LIYAB_REQUIRE(a != nullptr, "gemm_rows: null operand");
    if (int rc = check_rows(w, M, N, K, epi)) return rc;
    LIYAB_REQUIRE(al16(a) && lda % 8 == 0 && lda >= K, "gemm_rows: rows must be 16-byte aligned (row stride %lld)", static_cast<long long>(lda));
    if (M == 0) return 0;
    Source src{};
    src.a = static_cast<const bf16_t*>(a);
    src.lda = lda;
    return launch_epi<kRows>(src, static_cast<const bf16_t*>(w), M, N, K, strip, *epi, stream);
}

// The same over LayerNorm(x) of 32-bit rows x [M, K], K <= 2048.
extern "C" int liyab_gemm_rows_ln(const float* x, const float* ln_weight, const float* ln_bias, float eps, const void* w, int M, int N, int K,
                                  int strip, const EpiParams* epi, hipStream_t stream) {
    LIYAB_REQUIRE(x != nullptr, "gemm_rows_ln: null operand");
    if (int rc = check_rows(w, M, N, K, epi)) return rc;
    LIYAB_REQUIRE(K <= 2048 && eps >= 0.0f, "gemm_rows_ln: rows of %d (at most 2048), eps %g", K, static_cast<double>(eps));
    LIYAB_REQUIRE(al16(x) && al16(ln_weight) && al16(ln_bias), "gemm_rows_ln: operands must be 16-byte aligned");
    LIYAB_REQUIRE(epi->mode != kEpiResidual, "gemm_rows_ln: the residual epilogue is not taken");
    if (M == 0) return 0;
    Source src{};
    src.x = x;
    src.weight = ln_weight;
    src.bias = ln_bias;
    src.eps = eps;
    return launch_epi<kNorm>(src, static_cast<const bf16_t*>(w), M, N, K, strip, *epi, stream);
}

// residual += merge(partials) . w^T + bias over attention's splits [M][n_head][n_splits <= 8][hd + 4] (liyab_attention_decode with
// leave_splits), K = n_head * hd. The rows lie in LDS, up to 32 a workgroup: 32 of up to 2,240 fit whatever the strip, 8 of 8,192; what does not is refused.
extern "C" int liyab_gemm_rows_splits(const float* partials, int n_splits, int n_head, int hd, const void* w, int M, int N, int strip,
                                      const EpiParams* epi, hipStream_t stream) {
    LIYAB_REQUIRE(partials != nullptr, "gemm_rows_splits: null operand");
    LIYAB_REQUIRE(n_splits >= 1 && n_splits <= 8 && n_head > 0 && hd > 0 && hd % 4 == 0 && static_cast<int64_t>(n_head) * hd <= 8192,
                  "gemm_rows_splits: %d splits (1 to 8) of %d heads of %d", n_splits, n_head, hd);
    if (int rc = check_rows(w, M, N, n_head * hd, epi)) return rc;
    LIYAB_REQUIRE(al16(partials) && epi->mode == kEpiResidual, "gemm_rows_splits: 16-byte aligned splits, and the residual epilogue");
    if (M == 0) return 0;
    Source src{};
    src.x = partials;
    src.n_splits = n_splits;
    src.n_head = n_head;
    src.hd = hd;
    return launch_epi<kSplits>(src, static_cast<const bf16_t*>(w), M, N, n_head * hd, strip, *epi, stream);
}
