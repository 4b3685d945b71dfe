// out[M,N] = a[M,K] . w[N,K]^T in bfloat16 on the matrix cores for many rows: tiles from 64 x 64 to 256 x 256, operands
// straight from global memory into a ring of stages in LDS (global_load_lds, 16 bytes a lane), 64 k a stage. K must be a
// multiple of 64.
//
// What bounds it. The matrix cores draw more power than the card has: on random data, nothing but products, 32 x 32 x 16
// instructions settle at 1.6-1.8 PFLOP/s and 16 x 16 x 32 at 1.9-2.1 (2.4 on zeros), so the blocks are 16 x 16. A compute unit
// takes operands in at about 113 GB/s, loads alone, when a load covers whole lines of 128 bytes, and at 70 when it covers
// halves of them (stages of 32 k), so a stage is 64 k. Beside the loads LDS hands the fragments out, 128 bytes a cycle: of the small tiles that is the larger
// part (a stage of 64 x 64: 384 cycles of LDS, 128 of products), and then a chain of barrier, reads and products whose length the reads' latency sets: all of a
// stage's fragments are read at once (780 rows, 4,096 -> 1,024, cold weights: 22.8 us in halves, 20.7 at once; 400 rows of 1,024 -> 1,024 8.4 and 7.4). Of tiles
// whose waves would stand at the load queue the loads go out in two halves, each in front of the products of 32 k. What is left unhidden (a stage's barrier,
// the first fragments, the outputs) overlaps with another workgroup's products: two workgroups of eight waves a compute unit for the middle tiles; 256 x 256
// has eight waves or sixteen (launch_tile_256).
// Alone and repeated, 8,192 cubed ran at 1.32 PFLOP/s on sixteen waves (the vendor's library 1.44).
// Tried and left, cold weights: rings of six to nine stages for small tiles (no faster: not the latency of memory), fragments a stage or half of one ahead in
// registers of their own, strung between the products (3 to 30 % slower), some waves
// that load `a` only and others `w` (in steps 1 to 3 % slower), one wave a SIMD with parts of 96 x 64 to 128 x 128 (15 to 60 % slower); tiles of 128 x 64, 128 x
// 96, 128 x 160, 192 x 192, 256 x 128, 160 x 256, 256 x 192 and 160 x 320 under a model fitted to 232 products alone (4 % faster there on their average; in steps up to 3 % slower); rows of `w` and `a` 64 elements further apart (no change);
// bands of columns in the tiles' order, which bring fewer rows of `w` into an XCD's L2 (alone up to 8 % faster, in a step slower: the kernels around them find fewer of their rows there, 8,001 tokens
// 768 -> 2,304 40.8 -> 46.1). Faster,
// but with sums in another order, which moves a sampled token where two logits lie within the rounding: groups of waves that walk K side by side (64 x 64 and 64 x 96, 5 to 20 %
// with a compute unit a tile), XCDs that start an eighth of K apart (they ask for the same rows of `w` at once: 3,072 -> 768 of 2,048 rows 21.8 -> 18.8).
#include "common.h"
#include "launchers.h"
#include "gemm_tile.h"

namespace liyab {

typedef __attribute__((address_space(3))) void* lds_void_ptr;

constexpr int TBK = 64;  // k a stage

template <int BM, int BN, int STAGES, int WM, int WN>
constexpr size_t tile_lds_bytes(size_t out_bytes) {
    const size_t stages = static_cast<size_t>(STAGES) * (BM + BN) * TBK * 2, staging = staging_bytes<BM, BN, WM, WN, 1>(out_bytes);
    return stages > staging ? stages : staging;
}

// WM x WN waves, each with (BM / WM) x (BN / WN) of the tile in blocks of 16 x 16; MIN_WAVES a SIMD: what the registers must leave room for (the
// workgroups that LDS lets a compute unit hold). HALVES: a stage's loads and fragments in two halves of 32 k, for tiles whose waves ask for more than the
// load queue takes; otherwise all of a stage's fragments are read at once, ahead of its products and of the loads.
template <int BM, int BN, int STAGES, typename OutT, int EPI, int WM, int WN, int MIN_WAVES, bool HALVES>
__global__ void __launch_bounds__(64 * WM * WN, MIN_WAVES)
gemm_mfma_tile_kernel(const bf16_t* __restrict__ a, int64_t lda, const bf16_t* __restrict__ w, int M, int N, int K, EpiParams epi, int vec_ok,
                      int page_shift, PartsParams parts) {
    constexpr int WAVES = WM * WN, TM = BM / WM / 16, TN = BN / WN / 16, STAGE = (BM + BN) * TBK;
    constexpr int A_LOADS = BM / 8 / WAVES, W_LOADS = BN / 8 / WAVES, LOADS = A_LOADS + W_LOADS;  // 1 KiB each: 8 rows of 64 k
    static_assert(A_LOADS * 8 * WAVES == BM && W_LOADS * 8 * WAVES == BN, "whole loads a wave");
    static_assert(STAGES >= 2 && STAGES <= 4 && (STAGES - 2) * LOADS <= 63, "the waits below");
    extern __shared__ __attribute__((aligned(1024))) bf16_t lds[];
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int wm = wave / WN, wn = wave % WN;
    int m0, n0;
    tile_place<BM, BN>(M, N, K, m0, n0);

    int units = K / TBK, first = 0;  // units of k this workgroup walks, and where it starts
    if constexpr (EPI == kEpiParts) {
        first = blockIdx.y * parts.kt_per_part;
        units = min(units - first, parts.kt_per_part);
        if (blockIdx.y > 0) epi.bias = nullptr;  // the bias goes to the first plane only
    }
    // A load fills 1 KiB of LDS lane after lane: 8 rows of 128 bytes, unpadded. A 16-byte read serves 16 lanes a cycle, here 16
    // consecutive rows at one piece: even and odd rows start in different halves of the 64 banks, and within a half 8 rows
    // must land on 8 different pieces, so piece c of a row lies at c ^ ((row / 2) % 8). Rows past M or N: the last valid one
    // again; what comes of them is never stored.
    const bf16_t* src[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int row = (i < A_LOADS ? wave * A_LOADS + i : wave * W_LOADS + i - A_LOADS) * 8 + lane / 8;
        const int c = (lane % 8) ^ ((row >> 1) & 7);
        src[i] = (i < A_LOADS ? a + static_cast<int64_t>(min(m0 + row, M - 1)) * lda : w + static_cast<int64_t>(min(n0 + row, N - 1)) * K) + first * TBK + c * 8;
    }
    bf16_t* const to_a = lds + wave * A_LOADS * 512;
    bf16_t* const to_w = lds + BM * TBK + wave * W_LOADS * 512;
    auto issue = [&](int begin, int end, int unit, int stage) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            if (i < begin || i >= end) continue;
            const bf16_t* from = src[i] + unit * TBK;
            bf16_t* to = (i < A_LOADS ? to_a + i * 512 : to_w + (i - A_LOADS) * 512) + stage * STAGE;
            __builtin_amdgcn_global_load_lds(from, (lds_void_ptr)(to), 16, 0, 0);
        }
    };

    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const int li = lane % 16, g = lane / 16, swizzle = (li >> 1) & 7;  // (rows of a block start at multiples of 16)
    const int row_a = (wm * (BM / WM) + li) * TBK, row_w = BM * TBK + (wn * (BN / WN) + li) * TBK;
    struct Frags {
        bf16x8 a[TM], w[TN];
    };
    auto read = [&](Frags& f, int stage, int half) {  // 32 k
        const bf16_t* piece = lds + stage * STAGE + (((4 * half + g) ^ swizzle) * 8);
#pragma unroll
        for (int j = 0; j < TN; ++j) f.w[j] = *reinterpret_cast<const bf16x8*>(piece + row_w + j * 16 * TBK);
#pragma unroll
        for (int i = 0; i < TM; ++i) f.a[i] = *reinterpret_cast<const bf16x8*>(piece + row_a + i * 16 * TBK);
    };
    auto multiply = [&](const Frags& f) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.w[j], f.a[i], acc[i][j], 0, 0, 0);
    };

#pragma unroll
    for (int p = 0; p < STAGES - 1; ++p)
        if (p < units) issue(0, LOADS, p, p);
    for (int u = 0, stage = 0, next = STAGES - 1; u < units; ++u) {
        // stage u must have landed; the loads of the stages after it may be in flight (a wave's loads complete in order)
        const int later = min(units - 1 - u, STAGES - 2);
        if (STAGES > 3 && later >= 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(STAGES > 3 ? 2 * LOADS : 0) : "memory");
        else if (STAGES > 2 && later >= 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(STAGES > 2 ? LOADS : 0) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        // everyone's loads of stage u are in LDS, everyone is done reading stage u - 1: its place takes stage u + STAGES - 1
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        const bool more = u + STAGES - 1 < units;
        Frags f[2];
        if constexpr (HALVES) {
            if (more) issue(0, (LOADS + 1) / 2, u + STAGES - 1, next);
            read(f[0], stage, 0);
            multiply(f[0]);
            __builtin_amdgcn_sched_barrier(0);
            if (more) issue((LOADS + 1) / 2, LOADS, u + STAGES - 1, next);
            read(f[1], stage, 1);
            multiply(f[1]);
            __builtin_amdgcn_sched_barrier(0);
        } else {
            read(f[0], stage, 0);
            read(f[1], stage, 1);
            if (more) issue(0, LOADS, u + STAGES - 1, next);
            __builtin_amdgcn_sched_barrier(0);
            multiply(f[0]);
            multiply(f[1]);
            __builtin_amdgcn_sched_barrier(0);  // (its products, and with them the reads they wait for, stay ahead of the next barrier)
        }
        stage = stage + 1 == STAGES ? 0 : stage + 1;
        next = next + 1 == STAGES ? 0 : next + 1;
    }
    store_tile<BM, BN, OutT, EPI, WM, WN>(acc, lds, epi, parts, m0, n0, M, N, vec_ok, page_shift, wave, wm, wn, lane);
}

template <int BM, int BN, int STAGES, int WM, int WN, int MIN_WAVES, bool HALVES, typename OutT, int EPI>
int launch_tile_as(const bf16_t* a, int64_t lda, const bf16_t* w, int M, int N, int K, const EpiParams& epi, int kparts, const PartsParams& parts,
                   hipStream_t stream) {
    constexpr size_t smem = tile_lds_bytes<BM, BN, STAGES, WM, WN>(sizeof(OutT));
    static_assert(smem <= 160 * 1024, "a workgroup's LDS");
    auto kern = gemm_mfma_tile_kernel<BM, BN, STAGES, OutT, EPI, WM, WN, MIN_WAVES, HALVES>;
    static bool ready = false;  // once per instantiation, outside any stream capture's first use
    if (!ready) {
        hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(smem));
        ready = true;
    }
    int vec_ok, page_shift;
    store_rules<OutT, EPI>(epi, N, vec_ok, page_shift);
    if (EPI == kEpiParts && ((reinterpret_cast<uintptr_t>(parts.base) & 15) != 0 || parts.part_stride % 4 != 0 || parts.base_stride % 4 != 0)) vec_ok = 0;
    const dim3 grid(((N + BN - 1) / BN) * ((M + BM - 1) / BM), kparts);
    kern<<<grid, 64 * WM * WN, smem, stream>>>(a, lda, w, M, N, K, epi, vec_ok, page_shift, parts);
    return check_launch("gemm_mfma_tile");
}

// (each epilogue a kernel: one that chooses as it stores is too long a loop to unroll over 128 sums a lane, which then lie in memory)
#define LIYAB_TILE(T, E) launch_tile_as<BM, BN, STAGES, WM, WN, MIN_WAVES, HALVES, T, E>(a, lda, w, M, N, K, epi, 1, PartsParams{}, stream)
template <int BM, int BN, int STAGES, int WM, int WN, int MIN_WAVES, bool HALVES>
int launch_tile_gelu(const bf16_t* a, int64_t lda, const bf16_t* w, int M, int N, int K, const EpiParams& epi, hipStream_t stream) {
    const bool f32 = epi.out_dtype == kF32;
    if (epi.mode == kEpiGeluTanh) return f32 ? LIYAB_TILE(float, kEpiGeluTanh) : LIYAB_TILE(bf16_t, kEpiGeluTanh);
    return f32 ? LIYAB_TILE(float, kEpiGeluErf) : LIYAB_TILE(bf16_t, kEpiGeluErf);
}

template <int BM, int BN, int STAGES, int WM, int WN, int MIN_WAVES, bool HALVES>
int launch_tile_plain(const bf16_t* a, int64_t lda, const bf16_t* w, int M, int N, int K, const EpiParams& epi, hipStream_t stream) {
    const bool f32 = epi.out_dtype == kF32;
    switch (epi.mode) {
        case kEpiResidual: return LIYAB_TILE(float, kEpiResidual);
        case kEpiNone: return f32 ? LIYAB_TILE(float, kEpiNone) : LIYAB_TILE(bf16_t, kEpiNone);
        case kEpiQkvPaged: return f32 ? LIYAB_TILE(float, kEpiQkvPaged) : LIYAB_TILE(bf16_t, kEpiQkvPaged);
        default: return fail(1, "gemm: unknown epilogue %d", epi.mode);
    }
}
#undef LIYAB_TILE

inline bool is_gelu(const EpiParams& epi) { return epi.mode == kEpiGeluTanh || epi.mode == kEpiGeluErf; }

template <int BM, int BN, int STAGES, int WM, int WN, int MIN_WAVES, bool HALVES>
int launch_tile_epi(const bf16_t* a, int64_t lda, const bf16_t* w, int M, int N, int K, const EpiParams& epi, hipStream_t stream) {
    return is_gelu(epi) ? launch_tile_gelu<BM, BN, STAGES, WM, WN, MIN_WAVES, HALVES>(a, lda, w, M, N, K, epi, stream)
                        : launch_tile_plain<BM, BN, STAGES, WM, WN, MIN_WAVES, HALVES>(a, lda, w, M, N, K, epi, stream);
}

// 256 x 256. Eight waves of 128 x 64 read LDS less than sixteen of 64 x 64, which counts the more the longer K is; sixteen have twice as many at an activation's
// arithmetic, which two a SIMD don't hide. us, sixteen / eight, cold weights: 7,900 rows back to the stream, 1,600 -> 1,600 57.0 / 55.2, 4,096 -> 1,024 110.4 / 103.5, 6,400 ->
// 1,600 171 / 163; no activation, 1,600 -> 4,800 129.5 / 129.4, 1,024 -> 3,072 60.3 / 60.6; tanh, 1,600 -> 6,400 189.9 / 187.5, 2,048 -> 8,192 248 / 241, but 1,280 -> 5,120
// 122.0 / 122.5 and of 3,800 rows of 1,280 -> 3,840 44.3 / 44.9; erf, 1,600 -> 6,400 222 / 238, 1,024 -> 4,096 of 3,800 rows 47.3 / 51.6.
int launch_tile_256(const bf16_t* a, int64_t lda, const bf16_t* w, int M, int N, int K, const EpiParams& epi, hipStream_t stream) {
    if (epi.mode == kEpiGeluTanh && epi.out_dtype == kBF16 && K >= 1536)
        return launch_tile_as<256, 256, 2, 2, 4, 2, false, bf16_t, kEpiGeluTanh>(a, lda, w, M, N, K, epi, 1, PartsParams{}, stream);
    return is_gelu(epi) ? launch_tile_gelu<256, 256, 2, 4, 4, 4, true>(a, lda, w, M, N, K, epi, stream)
                        : launch_tile_plain<256, 256, 2, 2, 4, 2, false>(a, lda, w, M, N, K, epi, stream);
}

int choose_gemm_tile(int M, int N, int K) {
    // The compute units take tiles in rounds. A tile's time a unit of 64 k, measured alone on a compute unit and beside as many
    // others as fit there, and what a round costs besides (the first operands, the outputs, of which the single workgroup of a 256 x
    // 256 tile overlaps nothing), in us; a last round that is not full runs at the lower occupancy's time.
    struct Shape { int tile, bm, bn, fit; float unit[3], round; };
    constexpr Shape shapes[] = {
        {15, 256, 256, 1, {1.45f, 0, 0}, 10.0f}, {9, 192, 128, 2, {0.68f, 1.3f, 0}, 5.0f},  {11, 192, 128, 1, {0.62f, 0, 0}, 4.5f},
        {21, 128, 192, 1, {0.62f, 0, 0}, 4.5f},  {8, 128, 128, 2, {0.60f, 1.0f, 0}, 4.0f},  {7, 128, 128, 1, {0.50f, 0, 0}, 3.7f},
        {6, 64, 64, 2, {0.26f, 0.45f, 0}, 2.0f}, {2, 64, 64, 3, {0.30f, 0.45f, 0.62f}, 2.0f}};
    constexpr int kUnits = 256;  // compute units
    int best = 0;
    float best_us = 0.0f;
    for (const Shape& s : shapes) {
        const int64_t tiles = static_cast<int64_t>((M + s.bm - 1) / s.bm) * ((N + s.bn - 1) / s.bn);
        if (s.tile == 21 && tiles > kUnits) continue;
        const int64_t slots = static_cast<int64_t>(kUnits) * s.fit, full = tiles / slots, rest = tiles % slots;
        float us = full * (s.unit[s.fit - 1] * (K / TBK) + s.round);
        if (rest > 0) us += s.unit[(rest + kUnits - 1) / kUnits - 1] * (K / TBK) + s.round;
        if (best == 0 || us < best_us) {
            best = s.tile;
            best_us = us;
        }
    }
    // (256 x 256's times are those of sixteen waves: with the eight waves' own, 1.38 and 11, it took 6,148 to 7,100 rows of 2,048 -> 6,144 from 192 x 128, 154.2 us against 157.2 there at
    // 6,550 rows, 162.8 against 167.6 with tanh.)
    // 128 x 192 is here for products that it takes in one round and 128 x 128 in two: 250 to 256 tiles of it save 4 to 28 % (us, 128 x 128 / it, cold weights: 1,274 rows of
    // 1,600 -> 4,800 29.5 / 25.3, 2,015 of 768 -> 3,072 18.1 / 16.5, 8,125 of 3,072 -> 768 52.7 / 44.7, 4,095 of 512 -> 1,536 12.9 / 12.4). From the second round on, where
    // nothing overlaps a round's ends, it loses to all three that the times above put behind it (192 x 128: 7,740 rows of 1,600 -> 4,800 122 / 133, 8,115 of 768 -> 2,304 35.6 / 38.9;
    // 256 x 256: 2,515 of 1,600 -> 4,800 42.2 / 44.2; 128 x 128: 8,115 of 768 -> 3,072 49.3 / 56.2).
    // Tiles of 64 x 64 in three stages and in four cost nearly the same here. With a compute unit each, two on every unit, or a long K the fourth
    // stage is worth its LDS (780 rows, 5,120 -> 1,280 33.4 us against 35.2 in three; 361 rows, 1,280 -> 5,120 14.7 against 14.9); a round
    // in between with a short K takes three (512 rows: 768 -> 2,304 8.9 against 9.7, 1,024 -> 3,072 10.8 against 11.5).
    const int64_t small = static_cast<int64_t>((M + 63) / 64) * ((N + 63) / 64);
    if (best == 6 && K < 1280 && small > kUnits && small < 2 * kUnits) best = 2;
    return best;
}

int launch_gemm_tile(int tile, const bf16_t* a, int64_t lda, const bf16_t* w, int M, int N, int K, const EpiParams& epi, hipStream_t stream) {
    switch (tile) {
        case 2: return launch_tile_epi<64, 64, 3, 2, 2, 3, false>(a, lda, w, M, N, K, epi, stream);
        case 6: return launch_tile_epi<64, 64, 4, 2, 2, 2, false>(a, lda, w, M, N, K, epi, stream);
        case 7: return launch_tile_epi<128, 128, 3, 4, 2, 2, true>(a, lda, w, M, N, K, epi, stream);
        case 8: return launch_tile_epi<128, 128, 2, 4, 2, 4, true>(a, lda, w, M, N, K, epi, stream);
        case 9: return launch_tile_epi<192, 128, 2, 4, 2, 4, true>(a, lda, w, M, N, K, epi, stream);
        case 11: return launch_tile_epi<192, 128, 3, 4, 2, 2, true>(a, lda, w, M, N, K, epi, stream);
        case 15: return launch_tile_256(a, lda, w, M, N, K, epi, stream);
        case 21: return launch_tile_epi<128, 192, 3, 2, 4, 2, false>(a, lda, w, M, N, K, epi, stream);
        default: return fail(1, "gemm_mfma_dl: unknown tile %d", tile);
    }
}

int launch_gemm_tile_parts(const bf16_t* a, int64_t lda, const bf16_t* w, int M, int N, int K, int kparts, const EpiParams& epi, const PartsParams& parts,
                           hipStream_t stream) {
    return launch_tile_as<64, 64, 4, 2, 2, 2, false, float, kEpiParts>(a, lda, w, M, N, K, epi, kparts, parts, stream);
}

}  // namespace liyab
