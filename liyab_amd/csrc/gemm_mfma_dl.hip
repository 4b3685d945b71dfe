// out[M,N] = a[M,K] . w[N,K]^T in bfloat16 on the matrix cores, with tiles
// brought from global memory straight into LDS (global_load_lds, 16 bytes a
// lane) in a ring of three stages, so that two tiles of K are in flight
// while one is multiplied. For steps of many tokens; K must be a multiple of
// 64 (other shapes go to the register-staged kernel in gemm_mfma.hip). These
// are the tiles of few rows, whose groups of waves walk K side by side, and
// those of the batch-invariant mode; gemm_mfma_tile.hip has the others.
//
// A wave's direct load fills 1 KiB of LDS contiguously, lane after lane: 8
// rows of 64 k. Rows are therefore unpadded (128 bytes), and bank conflicts
// of the 16-byte fragment reads are avoided by a swizzle: within a row, the
// 16-byte piece c sits at position c ^ swizzle(row), applied on the
// global side when loading and again when reading. Rows past M or N are
// clamped to the last valid row; their results are never stored. MFMA
// operand layout and the fixed-order sum over k are those of gemm_mfma.hip.
//
// The product may be cut over K into parts (blockIdx.y), one plane of 32-bit
// sums a part, the first plane also taking the bias and the rows the product
// is added to (themselves a sum of planes): the planes together are then the
// residual stream after the product, as the streaming kernel of few rows
// leaves it (gemm_skinny.hip). A product with few output tiles and a long K
// covers the chip that way.
#include "common.h"
#include "launchers.h"
#include "gemm_tile.h"

#include <type_traits>

namespace liyab {

typedef __attribute__((address_space(3))) void* lds_void_ptr;

constexpr int DBK = 64;      // k per stage
// Where a row's 16-byte pieces sit within the row. LDS has 64 banks of 4 bytes: a 16-byte read
// serves 16 lanes a cycle, which read 16 consecutive rows at one piece index. Rows are 128 bytes,
// so even and odd rows start in different halves of the banks; within a half, 8 rows must land on
// 8 different pieces: the piece index is XORed with (row / 2) % 8.
__device__ __forceinline__ int swizzle(int row) { return (row >> 1) & 7; }

// Dynamic LDS of a workgroup: the operand stages, or, where bfloat16 outputs leave through LDS as whole
// rows, the waves' padded output tiles if those take more (tiles of 256 x 256: 144 KB against 128).
template <int BM, int BN, int DSTAGES, int WM, int WN, int WK>
constexpr size_t dl_lds_bytes(size_t out_bytes) {
    const size_t stages = static_cast<size_t>(DSTAGES) * WK * (BM + BN) * 64 * 2;
    const size_t staging = staging_bytes<BM, BN, WM, WN, WK>(out_bytes);
    return stages > staging ? stages : staging;
}

template <int BM, int BN, int DSTAGES, typename OutT, int EPI, int WM = 2, int WN = 2, int WK = 1, int SETS = 1>
__global__ void __launch_bounds__(64 * WM * WN * WK)
gemm_mfma_dl_kernel(const bf16_t* __restrict__ a, int64_t lda, const bf16_t* __restrict__ w, int M, int N, int K,
                    EpiParams epi, int vec_ok, int page_shift, PartsParams parts) {
    // WK groups of WM x WN waves, each wave with (BM / WM) x (BN / WN) of the tile in blocks of 32 x 32.
    // A stage holds WK consecutive units of 64 k, one a group: the groups walk K side by side (a
    // tile of few rows has few products a unit, and its walk is a chain of waits: load, barrier,
    // fragments, products; WK of them run at once), and their sums are added at the end in the
    // groups' order. SETS (with WK = 1): the one group keeps SETS sums, unit u of 64 k going to sum
    // u % SETS, added at the end in the sums' order: what WK = SETS groups would have left, bit
    // for bit, so that a row has one result in tiles of every shape (the batch-invariant mode).
    static_assert(SETS == 1 || (WK == 1 && SETS == 4), "sums by unit are for one group of waves, four of them");
    constexpr int GROUP = WM * WN, WAVES = GROUP * WK, TM = BM / WM / 32, TN = BN / WN / 32;
    constexpr int UNIT = (BM + BN) * DBK;       // elements of one unit of 64 k: the tile of a, then the tile of w
    constexpr int STAGE = WK * UNIT;            // elements per stage
    constexpr int A_LOADS = BM / 8 / GROUP, W_LOADS = BN / 8 / GROUP;  // wave-loads (8 rows each) per wave and stage
    static_assert(TM >= 1 && TN >= 1 && A_LOADS >= 1 && W_LOADS >= 1, "tile too small for its waves");
    extern __shared__ __attribute__((aligned(1024))) bf16_t lds[];

    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    const int wk = wave / GROUP, wg = wave % GROUP;
    const int wm = wg / WN, wn = wg % WN;
    int m0, n0;
    tile_place<BM, BN>(M, N, K, m0, n0);
    const int li = lane % 32, g = lane / 32;

    // this lane's part in a wave-load: row lane / 8 of the 8, LDS piece position lane % 8
    const int lrow = lane / 8, lpos = lane % 8;
    // a group's waves load their group's unit of the stage; a unit past the end of K is the last
    // one again (loaded and not multiplied: every wave asks for as many loads a stage as the
    // waits below count on)
    int units = K / DBK;  // units of 64 k this workgroup walks
    auto issue = [&](int kt, int stage) {
        const int k0 = min(kt * WK + wk, units - 1) * DBK;
        bf16_t* sa = lds + stage * STAGE + wk * UNIT;
        bf16_t* sw = sa + BM * DBK;
#pragma unroll
        for (int i = 0; i < A_LOADS; ++i) {
            const int r0 = (wg * A_LOADS + i) * 8, row = r0 + lrow;
            const int c = lpos ^ swizzle(row);
            const bf16_t* src = a + static_cast<int64_t>(min(m0 + row, M - 1)) * lda + k0 + c * 8;
            __builtin_amdgcn_global_load_lds(src, (lds_void_ptr)(sa + r0 * DBK), 16, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < W_LOADS; ++i) {
            const int r0 = (wg * W_LOADS + i) * 8, row = r0 + lrow;
            const int c = lpos ^ swizzle(row);
            const bf16_t* src = w + static_cast<int64_t>(min(n0 + row, N - 1)) * K + k0 + c * 8;
            __builtin_amdgcn_global_load_lds(src, (lds_void_ptr)(sw + r0 * DBK), 16, 0, 0);
        }
    };

    floatx16 sums[SETS][TM][TN];
#pragma unroll
    for (int s = 0; s < SETS; ++s)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) sums[s][i][j][r] = 0.0f;

    if constexpr (EPI == kEpiParts) {
        // this workgroup's part of K: units [kt0, kt0 + units)
        const int kt0 = blockIdx.y * parts.kt_per_part;
        units = min(units - kt0, parts.kt_per_part);
        a += static_cast<int64_t>(kt0) * DBK;
        w += static_cast<int64_t>(kt0) * DBK;
        if (blockIdx.y > 0) epi.bias = nullptr;  // the bias goes to the first plane only
    }
    const int nk = (units + WK - 1) / WK;  // stages walked
    constexpr int AHEAD = DSTAGES - 1;  // tiles of K in flight or in use beside the one being multiplied
#pragma unroll
    for (int p = 0; p < AHEAD; ++p)
        if (p < nk) issue(p, p);
    auto step = [&](int kt, auto set) {
        floatx16 (&acc)[TM][TN] = sums[decltype(set)::value];
        // tile kt must have landed: the loads of the tiles after it may still be in flight (a
        // wave's loads complete in order, A_LOADS + W_LOADS a tile)
        const int later = min(nk - 1 - kt, AHEAD - 1);
        constexpr int PER_TILE = A_LOADS + W_LOADS;
        static_assert((AHEAD - 1) * PER_TILE <= 63, "the counter of loads in flight has six bits");
        if (later >= 7) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(AHEAD > 7 ? 7 * PER_TILE : 0) : "memory");
        else if (later == 6) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(AHEAD > 6 ? 6 * PER_TILE : 0) : "memory");
        else if (later == 5) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(AHEAD > 5 ? 5 * PER_TILE : 0) : "memory");
        else if (later == 4) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(AHEAD > 4 ? 4 * PER_TILE : 0) : "memory");
        else if (later == 3) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(AHEAD > 3 ? 3 * PER_TILE : 0) : "memory");
        else if (later == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * (A_LOADS + W_LOADS)) : "memory");
        else if (later == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(A_LOADS + W_LOADS) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        // everyone's loads of tile kt are in LDS; everyone is done reading tile kt - 1. A bare
        // barrier: __syncthreads() would also wait for the loads still meant to be in flight.
        __builtin_amdgcn_s_barrier();
        if (kt + AHEAD < nk) issue(kt + AHEAD, (kt + AHEAD) % DSTAGES);  // into the stage tile kt - 1 used
        const bf16_t* sa = lds + (kt % DSTAGES) * STAGE + wk * UNIT;
        const bf16_t* sw = sa + BM * DBK;
        if (WK > 1 && kt * WK + wk >= units) return;  // this group's unit is past the end of K (the last stage only)
        // fragments of slab ks + 1 are read from LDS while slab ks multiplies
        bf16x8 fa[2][TM], fw[2][TN];
        auto read_frags = [&](int ks, int buf) {
            const int c = ks * 2 + g;  // the 16-byte piece of the row this lane needs
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const int row = wm * (BM / WM) + i * 32 + li;
                fa[buf][i] = *reinterpret_cast<const bf16x8*>(sa + row * DBK + ((c ^ swizzle(row)) * 8));
            }
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int row = wn * (BN / WN) + j * 32 + li;
                fw[buf][j] = *reinterpret_cast<const bf16x8*>(sw + row * DBK + ((c ^ swizzle(row)) * 8));
            }
        };
        read_frags(0, 0);
#pragma unroll
        for (int ks = 0; ks < DBK / 16; ++ks) {
            if (ks + 1 < DBK / 16) read_frags(ks + 1, (ks + 1) & 1);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fw[ks & 1][j], fa[ks & 1][i], acc[i][j], 0, 0, 0);
        }
    };
    if constexpr (SETS == 1) {
        for (int kt = 0; kt < nk; ++kt) step(kt, std::integral_constant<int, 0>{});
    } else {
        for (int kt = 0; kt < nk; kt += 4) {
            step(kt, std::integral_constant<int, 0>{});
            if (kt + 1 < nk) step(kt + 1, std::integral_constant<int, 1>{});
            if (kt + 2 < nk) step(kt + 2, std::integral_constant<int, 2>{});
            if (kt + 3 < nk) step(kt + 3, std::integral_constant<int, 3>{});
        }
#pragma unroll
        for (int q = 1; q < SETS; ++q)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) sums[0][i][j][r] += sums[q][i][j][r];
    }
    floatx16 (&acc)[TM][TN] = sums[0];
    if constexpr (WK > 1) {
        // the groups' sums, added in the groups' order by the first group, which alone stores:
        // the others go through the epilogue as a tile below the last row
        constexpr int PER_WAVE = TM * TN * 16 * 64;
        static_assert((WK - 1) * GROUP * PER_WAVE * 4 <= DSTAGES * STAGE * 2, "the groups' sums must fit the operand stages");
        float* red = reinterpret_cast<float*>(lds);
        __syncthreads();  // everyone is done reading the last operand stage
        if (wk > 0) {
            float* mine = red + ((wk - 1) * GROUP + wg) * PER_WAVE + lane;
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) mine[((i * TN + j) * 16 + r) * 64] = acc[i][j][r];
        }
        __syncthreads();
        if (wk == 0) {
#pragma unroll
            for (int q = 1; q < WK; ++q) {
                const float* theirs = red + ((q - 1) * GROUP + wg) * PER_WAVE + lane;
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
#pragma unroll
                        for (int r = 0; r < 16; ++r) acc[i][j][r] += theirs[((i * TN + j) * 16 + r) * 64];
            }
        } else {
            m0 = M;
        }
    }
    store_tile<BM, BN, OutT, EPI, WM, WN>(acc, lds, epi, parts, m0, n0, M, N, vec_ok, page_shift, wave, wm, wn, lane);
}

template <int BM, int BN, int DSTAGES, typename OutT, int EPI, int WM = 2, int WN = 2, int WK = 1, int SETS = 1>
int launch_dl_as(const bf16_t* a, int64_t lda, const bf16_t* w, int M, int N, int K, const EpiParams& epi, hipStream_t stream) {
    const int grid = ((N + BN - 1) / BN) * ((M + BM - 1) / BM);
    constexpr size_t smem = dl_lds_bytes<BM, BN, DSTAGES, WM, WN, WK>(sizeof(OutT));
    static_assert(smem <= 160 * 1024, "a workgroup's LDS");
    auto kern = gemm_mfma_dl_kernel<BM, BN, DSTAGES, OutT, EPI, WM, WN, WK, SETS>;
    static bool ready = false;  // once per instantiation, outside any stream capture's first use
    if (!ready) {
        hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(smem));
        ready = true;
    }
    int vec_ok, page_shift;
    store_rules<OutT, EPI>(epi, N, vec_ok, page_shift);
    kern<<<grid, 64 * WM * WN * WK, smem, stream>>>(a, lda, w, M, N, K, epi, vec_ok, page_shift, PartsParams{});
    return check_launch("gemm_mfma_dl");
}

// The product cut over K into `kparts` parts (see the head of this file); epi carries the planes
// (out, float32, rows of N) and the first plane's bias.
template <int BM, int BN, int DSTAGES, int WM = 2, int WN = 2, int WK = 1>
int launch_dl_parts(const bf16_t* a, int64_t lda, const bf16_t* w, int M, int N, int K, int kparts, const EpiParams& epi,
                    const PartsParams& parts, hipStream_t stream) {
    const dim3 grid(((N + BN - 1) / BN) * ((M + BM - 1) / BM), kparts);
    const size_t smem = static_cast<size_t>(DSTAGES) * WK * (BM + BN) * DBK * sizeof(bf16_t);
    auto kern = gemm_mfma_dl_kernel<BM, BN, DSTAGES, float, kEpiParts, WM, WN, WK>;
    static bool ready = false;
    if (!ready) {
        hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(smem));
        ready = true;
    }
    auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    const bool vec = N % 4 == 0 && al16(epi.bias) && al16(epi.out) && al16(parts.base) && parts.part_stride % 4 == 0 && parts.base_stride % 4 == 0;
    kern<<<grid, 64 * WM * WN * WK, smem, stream>>>(a, lda, w, M, N, K, epi, vec ? 1 : 0, -1, parts);
    return check_launch("gemm_mfma_dl_parts");
}

template <int BM, int BN, int DSTAGES, int WM = 2, int WN = 2, int WK = 1, int SETS = 1>
int launch_dl(const void* a, int64_t lda, const void* w, int M, int N, int K, const EpiParams& epi, hipStream_t stream) {
    auto* pa = static_cast<const bf16_t*>(a);
    auto* pw = static_cast<const bf16_t*>(w);
    if (epi.mode == kEpiResidual) return launch_dl_as<BM, BN, DSTAGES, float, kEpiResidual, WM, WN, WK, SETS>(pa, lda, pw, M, N, K, epi, stream);
    if (epi.out_dtype == kF32) {
        if (epi.mode == kEpiNone) return launch_dl_as<BM, BN, DSTAGES, float, kEpiNone, WM, WN, WK, SETS>(pa, lda, pw, M, N, K, epi, stream);
        return launch_dl_as<BM, BN, DSTAGES, float, -1, WM, WN, WK, SETS>(pa, lda, pw, M, N, K, epi, stream);
    }
    switch (epi.mode) {
        case kEpiNone: return launch_dl_as<BM, BN, DSTAGES, bf16_t, kEpiNone, WM, WN, WK, SETS>(pa, lda, pw, M, N, K, epi, stream);
        case kEpiGeluTanh: return launch_dl_as<BM, BN, DSTAGES, bf16_t, kEpiGeluTanh, WM, WN, WK, SETS>(pa, lda, pw, M, N, K, epi, stream);
        case kEpiGeluErf: return launch_dl_as<BM, BN, DSTAGES, bf16_t, kEpiGeluErf, WM, WN, WK, SETS>(pa, lda, pw, M, N, K, epi, stream);
        case kEpiQkvPaged: return launch_dl_as<BM, BN, DSTAGES, bf16_t, kEpiQkvPaged, WM, WN, WK, SETS>(pa, lda, pw, M, N, K, epi, stream);
        default: return fail(1, "gemm: unknown epilogue %d", epi.mode);
    }
}

}  // namespace liyab

using namespace liyab;

// tile: 2, 6 to 9, 11, 15, 21 = from 64x64 to 256x256 (gemm_tile.h lists them; gemm_mfma_tile.hip also chooses
// among them for 0); 17 = 32x32 on four waves that walk K side by side (a workgroup then brings in a
// third less of the operands, and twice as many workgroups pull: 64 rows with cold weights, 768 -> 2,304 in
// 5.05 us against 5.53, 1,024 -> 3,072 in 5.97 against 6.85; for as long as every tile has a compute unit
// of its own: 1,600 -> 4,800 in 13.9 against 9.7); 16 = 64x32 on four groups of two waves that walk K side by side, three stages of
// four units (for one tile of rows: 8.2 us for 64 x 4,800 x 1,600 where two waves walking K alone, four
// stages deep, took 10.3; deeper rings for those took longer, 11.1 with eight stages: the walk waits on
// its own chain of load, barrier, fragments and products, not on the loads in flight); 18 = the same bits for up to 64 rows from waves
// with rings of their own (gemm_mfma_waves.hip; more rows than 64 are taken tile by tile).
extern "C" int liyab_gemm_mfma_dl(const void* a, int64_t lda, const void* w, int M, int N, int K, int tile,
                                  const EpiParams* epi_in, hipStream_t stream) {
    LIYAB_REQUIRE(a && w && epi_in, "gemm: null operand");
    LIYAB_REQUIRE(M > 0 && N > 0 && K > 0, "gemm_mfma_dl: bad sizes M=%d N=%d K=%d", M, N, K);
    LIYAB_REQUIRE(K % DBK == 0 && lda % 8 == 0 && lda >= K, "gemm_mfma_dl: K %d must be a multiple of 64 and lda %lld of 8", K,
                  static_cast<long long>(lda));
    LIYAB_REQUIRE((reinterpret_cast<uintptr_t>(a) & 15) == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0,
                  "gemm_mfma_dl: operands must be 16-byte aligned");
    EpiParams epi = *epi_in;
    if (int rc = check_epilogue(epi, M, N)) return rc;
    if (tile == 0) tile = choose_gemm_tile(M, N, K);
    switch (tile) {
        case 16: return launch_dl<64, 32, 3, 2, 1, 4>(a, lda, w, M, N, K, epi, stream);
        case 17: return launch_dl<32, 32, 3, 1, 1, 4>(a, lda, w, M, N, K, epi, stream);
        case 18: return launch_gemm_waves(static_cast<const bf16_t*>(a), lda, static_cast<const bf16_t*>(w), M, N, K, epi, 1, nullptr, stream);
        // 102, 106, 108: tiles of 64 x 64 and 128 x 128 with four sums by unit of K, whose results are those of 16 and 17 bit for bit
        case 102: return launch_dl<64, 64, 3, 2, 2, 1, 4>(a, lda, w, M, N, K, epi, stream);
        case 106: return launch_dl<64, 64, 4, 2, 2, 1, 4>(a, lda, w, M, N, K, epi, stream);
        case 108: return launch_dl<128, 128, 2, 4, 2, 1, 4>(a, lda, w, M, N, K, epi, stream);
        default: return launch_gemm_tile(tile, static_cast<const bf16_t*>(a), lda, static_cast<const bf16_t*>(w), M, N, K, epi, stream);
    }
}

// The same product cut over K: parts[p * part_stride + m * N + n] = sum over the p-th of `kparts` parts
// of K (whole tiles of 64) of a[m, k] w[n, k]. With `base` (n_base planes [M, N], base_stride floats
// apart, not overlapping `parts`) the first plane also takes bias[n] and base[0] + base[1] + ...;
// without it `bias` must be null. tile: 6 = 64x64 tiles, 16 = 64x32 (for one tile of rows), 17 = 32x32, 18 = gemm_mfma_waves.hip.
extern "C" int liyab_gemm_mfma_dl_parts(const void* a, int64_t lda, const void* w, int M, int N, int K, int kparts, int tile,
                                        float* parts, int64_t part_stride, const float* bias, const float* base, int n_base,
                                        int64_t base_stride, hipStream_t stream) {
    LIYAB_REQUIRE(a && w && parts, "gemm: null operand");
    LIYAB_REQUIRE(M > 0 && N > 0 && K > 0, "gemm_mfma_dl_parts: bad sizes M=%d N=%d K=%d", M, N, K);
    LIYAB_REQUIRE(K % DBK == 0 && lda % 8 == 0 && lda >= K, "gemm_mfma_dl_parts: K %d must be a multiple of 64 and lda %lld of 8", K,
                  static_cast<long long>(lda));
    LIYAB_REQUIRE((reinterpret_cast<uintptr_t>(a) & 15) == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0,
                  "gemm_mfma_dl_parts: operands must be 16-byte aligned");
    const int nk = K / DBK;
    LIYAB_REQUIRE(kparts >= 1 && kparts <= 16 && (kparts - 1) * ((nk + kparts - 1) / kparts) < nk,
                  "gemm_mfma_dl_parts: K = %d does not cut into %d parts of whole tiles of 64", K, kparts);
    LIYAB_REQUIRE(kparts == 1 || part_stride >= static_cast<int64_t>(M) * N, "gemm_mfma_dl_parts: planes of %lld overlap",
                  static_cast<long long>(part_stride));
    LIYAB_REQUIRE(base != nullptr || bias == nullptr, "gemm_mfma_dl_parts: a bias needs the rows it is added to");
    if (base != nullptr) {
        LIYAB_REQUIRE(n_base >= 1 && n_base <= 16 && (n_base == 1 || base_stride >= static_cast<int64_t>(M) * N),
                      "gemm_mfma_dl_parts: bad planes of rows to add to (%d, %lld apart)", n_base, static_cast<long long>(base_stride));
        const float* base_end = base + (n_base - 1) * base_stride + static_cast<int64_t>(M) * N;
        const float* parts_end = parts + (kparts - 1) * part_stride + static_cast<int64_t>(M) * N;
        LIYAB_REQUIRE(base_end <= parts || parts_end <= base, "gemm_mfma_dl_parts: the rows to add to overlap the planes written");
    }
    EpiParams epi{};
    epi.mode = kEpiNone;
    epi.out_dtype = kF32;
    epi.out = parts;
    epi.ldo = N;
    epi.bias = bias;
    const PartsParams pp{(nk + kparts - 1) / kparts, part_stride, base, n_base, base_stride};
    auto* pa = static_cast<const bf16_t*>(a);
    auto* pw = static_cast<const bf16_t*>(w);
    if (tile == 6) return launch_gemm_tile_parts(pa, lda, pw, M, N, K, kparts, epi, pp, stream);
    if (tile == 16) return launch_dl_parts<64, 32, 3, 2, 1, 4>(pa, lda, pw, M, N, K, kparts, epi, pp, stream);
    if (tile == 17) return launch_dl_parts<32, 32, 3, 1, 1, 4>(pa, lda, pw, M, N, K, kparts, epi, pp, stream);
    if (tile == 18) return launch_gemm_waves(pa, lda, pw, M, N, K, epi, kparts, &pp, stream);
    return fail(1, "gemm_mfma_dl_parts: unknown tile %d (6, 16, 17 or 18)", tile);
}
