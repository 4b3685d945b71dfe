// out[M,N] = a[M,K] . w[N,K]^T in bfloat16 for 17 to 64 rows (a step of so many requests), the bits of gemm_mfma_dl.hip's tiles 16 and 17: unit u of 64 k goes to sum
// u % 4, 16 k an instruction of 32 x 32, the four sums added in their order. A workgroup takes RB rows and NB features, its four waves a sum each, all rows and
// features of it, through a ring in LDS of the wave's own (ring.h). K must be a multiple of 64.
//
// What bounds it: not the weights' bytes (1,600 -> 4,800 is 15 MB, 3 us) but a compute unit's intake of both operands, 300 KB a workgroup of 64 x 32 at some 110
// GB/s, behind a cold start of 3 us. Those tiles' waves share a stage's rows and stand at a barrier between its arrival and its products, seven in a row; here a wave waits
// for its own loads by their count, and a place is asked for again as soon as it has been read. Two units in flight a wave are enough (three and four the same to 10 % slower: two workgroups of
// 32 x 32 with two share a compute unit). us, cold weights, those tiles / here: 64 rows 1,600 -> 4,800 10.4 / 8.9, -> 6,400 11.3 / 9.4, 1,280 -> 5,120 9.5 / 7.6, 1,024 -> 3,072 6.6 /
// 5.0, 768 -> 3,072 6.1 / 4.5, 6,400 -> 1,600 in four parts 12.4 / 9.6, 3,072 -> 768 in four 7.0 / 4.7; 48 rows 9.5 / 8.2, 9.8 / 8.7, 8.7 / 7.2, 6.4 / 4.8, 5.9 / 4.4, 11.6 / 9.4, 6.8 / 4.6;
// 24 rows 1,600 -> 4,800 8.2 / 6.7, 4,096 -> 4,096 13.2 / 10.3.
// Measured and left: eight waves and sums a workgroup in blocks of 16 x 16 (0 to 10 % slower than four, and other bits), thirteen (slower still); workgroups that start at
// different k (a remainder worked out at the start, 0.5 us, and no gain behind it).
#include "common.h"
#include "launchers.h"
#include "gemm_tile.h"
#include "ring.h"

namespace liyab {

constexpr int kWaveUnit = 64, kWaveSums = 4;

// Floats between the rows of a sum in LDS: four more than a row has, so that rows start in different banks.
template <int NB>
constexpr int kSumRow = NB + 4;
template <int RB, int NB, int R>
constexpr size_t waves_lds_bytes() {
    constexpr size_t ring = size_t(kWaveSums) * R * (RB + NB) * kWaveUnit * 2, sums = size_t(kWaveSums) * RB * kSumRow<NB> * 4;
    return ring > sums ? ring : sums;
}

template <int RB, int NB, int R, typename OutT, int EPI>
__global__ void __launch_bounds__(64 * kWaveSums)
gemm_waves_kernel(const bf16_t* __restrict__ a, int64_t lda, const bf16_t* __restrict__ w, int M, int N, int K, EpiParams epi, int vec_ok, int page_shift,
                  PartsParams parts) {
    constexpr int TM = (RB + 31) / 32, LOADS = (NB + RB) / 8, SLOT = (NB + RB) * kWaveUnit, QUADS = NB / 4, ROW = kSumRow<NB>;
    constexpr int EACH = (RB * QUADS + 255) / 256;  // outputs, four side by side, a thread
    static_assert((NB == 16 || NB == 32) && RB % 16 == 0 && RB <= 64 && (R - 1) * LOADS <= 63, "one block of features, the counter of loads in flight has six bits");
    extern __shared__ __attribute__((aligned(1024))) bf16_t waves_lds[];
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int li = lane % 32, g = lane / 32, n0 = blockIdx.x * NB, m0 = blockIdx.z * RB;
    int units = K / kWaveUnit;
    if constexpr (EPI == kEpiParts) {
        const int first = blockIdx.y * parts.kt_per_part;
        units = min(units - first, parts.kt_per_part);
        a += static_cast<int64_t>(first) * kWaveUnit;
        w += static_cast<int64_t>(first) * kWaveUnit;
        if (blockIdx.y > 0) epi.bias = nullptr;  // the bias goes to the first plane only
    }
    const int mine = (units - wave + kWaveSums - 1) / kWaveSums;  // this wave's units: wave, wave + 4, ...
    bf16_t* const ring = waves_lds + wave * R * SLOT;
    const int lrow = lane / 8, lpos = lane % 8;  // this lane's part in a load: 8 rows of 64 k
    const bf16_t* from[LOADS];
#pragma unroll
    for (int l = 0; l < LOADS; ++l) {
        const int row = 8 * l + lrow, c = (lpos ^ ring_swizzle(row)) * 8;  // (a's rows start at a multiple of 16: the same places)
        from[l] = (l < NB / 8 ? w + static_cast<int64_t>(min(n0 + row, N - 1)) * K : a + static_cast<int64_t>(min(m0 + row - NB, M - 1)) * lda) + c;
    }
    auto load = [&](int j, int slot) {  // unit j of this wave's (one past its last: the last of K, not multiplied)
        const int k = min(wave + kWaveSums * j, units - 1) * kWaveUnit;
#pragma unroll
        for (int l = 0; l < LOADS; ++l) {
            const bf16_t* const piece = from[l] + k;
            __builtin_amdgcn_global_load_lds(piece, (lds_void_ptr)(ring + slot * SLOT + l * 8 * kWaveUnit), 16, 0, 0);
        }
    };
#pragma unroll
    for (int p = 0; p < R; ++p) load(p, p);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");

    floatx16 acc[TM];
#pragma unroll
    for (int s = 0; s < TM; ++s)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[s][r] = 0.0f;
    auto multiply = [&](int slot) {
        const bf16_t* const at = ring + slot * SLOT;
        bf16x8 x[4], y[TM][4];
#pragma unroll
        for (int h = 0; h < 4; ++h) {
            x[h] = *reinterpret_cast<const bf16x8*>(at + (li % NB) * kWaveUnit + ((2 * h + g) ^ ring_swizzle(li % NB)) * 8);
#pragma unroll
            for (int s = 0; s < TM; ++s) {
                const int row = NB + min(32 * s + li, RB - 1);  // (rows past the workgroup's: the last again, not stored)
                y[s][h] = *reinterpret_cast<const bf16x8*>(at + row * kWaveUnit + ((2 * h + g) ^ ring_swizzle(row)) * 8);
            }
        }
#pragma unroll
        for (int h = 0; h < 4; ++h)
#pragma unroll
            for (int s = 0; s < TM; ++s) acc[s] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[h], y[s][h], acc[s], 0, 0, 0);
    };
    int j0 = 0;
    for (; j0 + R < mine; j0 += R)
        in_turn(std::make_integer_sequence<int, R>{}, [&](auto at) {
            constexpr int t = decltype(at)::value;
            wait_loads<(R - 1) * LOADS>();
            multiply(t);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the place has been read
            load(j0 + R + t, t);
        });
    in_turn(std::make_integer_sequence<int, R>{}, [&](auto at) {
        constexpr int t = decltype(at)::value;
        wait_loads<(R - 1 - t) * LOADS>();
        if (j0 + t < mine) multiply(t);
    });
    // what the epilogue adds is asked for while the sums go through LDS
    const bool based = EPI == kEpiParts && blockIdx.y == 0 && parts.base != nullptr;
    f32x4 bias[EACH], add[EACH];
#pragma unroll
    for (int t = 0; t < EACH; ++t) {
        const int e = tid + 256 * t, m = min(m0 + e / QUADS, M - 1), n = max(min(n0 + e % QUADS * 4, N - 4), 0);
        bias[t] = add[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        if (EPI < 0 || !vec_ok) continue;
        if (epi.bias != nullptr) bias[t] = *reinterpret_cast<const f32x4*>(epi.bias + n);
        if constexpr (EPI == kEpiResidual) add[t] = *reinterpret_cast<const f32x4*>(epi.residual + static_cast<int64_t>(m) * epi.ldr + n);
        if (based) {
            const float* const bp = parts.base + static_cast<int64_t>(m) * N + n;
            f32x4 plane[4];
#pragma unroll
            for (int p = 0; p < 4; ++p) plane[p] = *reinterpret_cast<const f32x4*>(bp + min(p, parts.n_base - 1) * parts.base_stride);
            add[t] = plane[0];
#pragma unroll
            for (int p = 1; p < 4; ++p)
                if (p < parts.n_base) add[t] += plane[p];
            for (int p = 4; p < parts.n_base; ++p) add[t] += *reinterpret_cast<const f32x4*>(bp + p * parts.base_stride);
        }
    }
    lds_barrier();  // (the sums take the rings' place)
    float* const red = reinterpret_cast<float*>(waves_lds);
    // acc[s][r]: row 32 s + li, feature 8 (r / 4) + 4 g + r % 4
#pragma unroll
    for (int s = 0; s < TM; ++s)
#pragma unroll
        for (int q = 0; q < NB / 8; ++q)
            if (RB % 32 == 0 || 32 * s + li < RB)
                *reinterpret_cast<f32x4*>(red + (wave * RB + 32 * s + li) * ROW + 8 * q + 4 * g) = f32x4{acc[s][4 * q], acc[s][4 * q + 1], acc[s][4 * q + 2], acc[s][4 * q + 3]};
    lds_barrier();
#pragma unroll
    for (int t = 0; t < EACH; ++t) {
        const int e = tid + 256 * t, m = m0 + e / QUADS, n = n0 + e % QUADS * 4;
        if (e >= RB * QUADS || m >= M || n >= N) continue;
        const float* const sums = red + (e / QUADS) * ROW + e % QUADS * 4;
        f32x4 v = *reinterpret_cast<const f32x4*>(sums);
#pragma unroll
        for (int q = 1; q < kWaveSums; ++q) v += *reinterpret_cast<const f32x4*>(sums + q * RB * ROW);
        if (EPI >= 0 && vec_ok) {  // (N is a multiple of 4)
            v += bias[t];
            if constexpr (EPI == kEpiParts) {
                *reinterpret_cast<f32x4*>(static_cast<float*>(epi.out) + blockIdx.y * parts.part_stride + static_cast<int64_t>(m) * N + n) = v + add[t];
            } else if constexpr (EPI == kEpiResidual) {
                *reinterpret_cast<f32x4*>(epi.residual + static_cast<int64_t>(m) * epi.ldr + n) = v + add[t];
            } else if constexpr (EPI == kEpiQkvPaged) {
                if (n < epi.q_dim) {
                    store4<OutT>(static_cast<OutT*>(epi.out) + static_cast<int64_t>(m) * epi.ldo + n, v);
                } else {
                    const int word = epi.slots[m];
                    const int page = page_shift >= 0 ? word >> page_shift : word / epi.page_size, off = word - page * epi.page_size;
                    if (static_cast<uint32_t>(word) >= epi.num_slots) continue;
                    const bool is_v = n >= epi.q_dim + epi.kv_dim;
                    const int c = n - epi.q_dim - (is_v ? epi.kv_dim : 0), head = c / epi.hd;
                    store4<OutT>(static_cast<OutT*>(is_v ? epi.vc : epi.kc) + ((static_cast<int64_t>(page) * epi.n_kv_head + head) * epi.page_size + off) * epi.hd + (c - head * epi.hd), v);
                }
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if constexpr (EPI == kEpiGeluTanh) v[r] = gelu_tanh_fast(v[r]);
                    if constexpr (EPI == kEpiGeluErf) v[r] = gelu_erf_fast(v[r]);
                }
                store4<OutT>(static_cast<OutT*>(epi.out) + static_cast<int64_t>(m) * epi.ldo + n, v);
            }
            continue;
        }
#pragma unroll 1
        for (int r = 0; r < 4 && n + r < N; ++r) {
            const float x = sums[r] + sums[RB * ROW + r] + sums[2 * RB * ROW + r] + sums[3 * RB * ROW + r];
            if constexpr (EPI == kEpiParts) {
                float y = x + epilogue_bias(epi, n + r);
                if (based) {
                    const float* const bp = parts.base + static_cast<int64_t>(m) * N + n + r;
                    float b = bp[0];
                    for (int p = 1; p < parts.n_base; ++p) b += bp[p * parts.base_stride];
                    y += b;
                }
                (static_cast<float*>(epi.out) + blockIdx.y * parts.part_stride)[static_cast<int64_t>(m) * N + n + r] = y;
            } else {
                epilogue_store<OutT, EPI, false>(epi, m, n + r, x);
            }
        }
    }
}

template <int RB, int NB, int R, typename OutT, int EPI>
int launch_waves_as(const bf16_t* a, int64_t lda, const bf16_t* w, int M, int N, int K, const EpiParams& epi, int kparts, const PartsParams& parts, hipStream_t stream) {
    constexpr size_t smem = waves_lds_bytes<RB, NB, R>();
    static_assert(smem <= 160 * 1024, "a workgroup's LDS");
    auto kern = gemm_waves_kernel<RB, NB, R, OutT, EPI>;
    static bool ready = false;  // once per instantiation, outside any stream capture's first use
    if (!ready) {
        hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(smem));
        ready = true;
    }
    int vec_ok, page_shift;
    store_rules<OutT, EPI>(epi, N, vec_ok, page_shift);
    if (EPI == kEpiParts && ((reinterpret_cast<uintptr_t>(parts.base) & 15) != 0 || parts.part_stride % 4 != 0 || parts.base_stride % 4 != 0)) vec_ok = 0;
    kern<<<dim3((N + NB - 1) / NB, kparts, (M + RB - 1) / RB), 64 * kWaveSums, smem, stream>>>(a, lda, w, M, N, K, epi, vec_ok, page_shift, parts);
    return check_launch("gemm_waves");
}

template <int RB, int NB>
int launch_waves_epi(const bf16_t* a, int64_t lda, const bf16_t* w, int M, int N, int K, const EpiParams& epi, int kparts, const PartsParams* parts, hipStream_t stream) {
#define LIYAB_WAVES(T, E) launch_waves_as<RB, NB, 2, T, E>(a, lda, w, M, N, K, epi, kparts, parts != nullptr ? *parts : PartsParams{}, stream)
    if (parts != nullptr) return LIYAB_WAVES(float, kEpiParts);
    if (epi.mode == kEpiResidual) return LIYAB_WAVES(float, kEpiResidual);
    if (epi.out_dtype == kF32) return epi.mode == kEpiNone ? LIYAB_WAVES(float, kEpiNone) : LIYAB_WAVES(float, -1);
    switch (epi.mode) {
        case kEpiNone: return LIYAB_WAVES(bf16_t, kEpiNone);
        case kEpiGeluTanh: return LIYAB_WAVES(bf16_t, kEpiGeluTanh);
        case kEpiGeluErf: return LIYAB_WAVES(bf16_t, kEpiGeluErf);
        case kEpiQkvPaged: return LIYAB_WAVES(bf16_t, kEpiQkvPaged);
        default: return fail(1, "gemm: unknown epilogue %d", epi.mode);
    }
#undef LIYAB_WAVES
}

int launch_gemm_waves(const bf16_t* a, int64_t lda, const bf16_t* w, int M, int N, int K, const EpiParams& epi, int kparts, const PartsParams* parts, hipStream_t stream) {
    // The smallest workgroups of which every compute unit takes one (us at 64 rows, 32 x 16 / 32 x 32 / 64 x 32: 1,024 -> 2,048 4.1 / 4.4 / -, 768 -> 2,304 4.3 / 3.7 / 4.7), 32 x 32 of
    // short walks and of parts also where some take two (1,280 -> 5,120 - / 7.6 / 8.1, 6,400 -> 1,600 in four parts - / 9.6 / 10.3; but 1,600 -> 4,800 - / 9.3 / 8.9), and
    // then all rows in one, so that the weights come in once (48 rows, 1,600 -> 6,400 in 48 x 32 8.7, in 32 x 32 9.2; 24 rows, 4,800 in 32 x 16 8.0, in 32 x 32 6.7).
    auto groups = [&](int rows, int features) { return static_cast<int64_t>((M + rows - 1) / rows) * ((N + features - 1) / features) * kparts; };
    if (groups(32, 16) <= 256) return launch_waves_epi<32, 16>(a, lda, w, M, N, K, epi, kparts, parts, stream);
    if (M <= 32 || groups(32, 32) <= (K <= 1280 || kparts > 1 ? 400 : 256)) return launch_waves_epi<32, 32>(a, lda, w, M, N, K, epi, kparts, parts, stream);
    if (M <= 48) return launch_waves_epi<48, 32>(a, lda, w, M, N, K, epi, kparts, parts, stream);
    return launch_waves_epi<64, 32>(a, lda, w, M, N, K, epi, kparts, parts, stream);
}

}  // namespace liyab
