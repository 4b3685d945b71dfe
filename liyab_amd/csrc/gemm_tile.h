// What the tiled matrix-core products share: which tile a workgroup takes, and how a wave's accumulators leave.
#pragma once

#include "common.h"
#include "epilogue.h"

#include <type_traits>

namespace liyab {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(16))) float floatx16;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((ext_vector_type(4))) float f32x4;

// Four consecutive outputs in one store (16 bytes of float32, 8 of bfloat16).
template <typename OutT>
__device__ __forceinline__ void store4(OutT* dst, const f32x4& v);
template <>
__device__ __forceinline__ void store4<float>(float* dst, const f32x4& v) { *reinterpret_cast<f32x4*>(dst) = v; }
template <>
__device__ __forceinline__ void store4<bf16_t>(bf16_t* dst, const f32x4& v) {
    uint2 packed;
    packed.x = static_cast<uint32_t>(float_to_bf16(v[0])) | (static_cast<uint32_t>(float_to_bf16(v[1])) << 16);
    packed.y = static_cast<uint32_t>(float_to_bf16(v[2])) | (static_cast<uint32_t>(float_to_bf16(v[3])) << 16);
    *reinterpret_cast<uint2*>(dst) = packed;
}

constexpr int kEpiParts = 5;  // the tiled products' own epilogue: a plane of sums a part of K

// A product cut over K: tiles of K a part, floats between the planes, and what the first plane adds.
struct PartsParams {
    int kt_per_part;
    int64_t part_stride;
    const float* base;  // rows the product is added to, a sum of n_base planes [M, N]; or null
    int n_base;
    int64_t base_stride;
};

// The tile of BM x BN that this workgroup (of gridDim.x, one a tile) takes: its first row and column.
template <int BM, int BN>
__device__ __forceinline__ void tile_place(int M, int N, int K, int& m0, int& n0) {
    // Workgroups go to the 8 XCDs round-robin, each XCD with an L2 of its own. Tile t of the
    // row-major tile order goes to the XCD that holds the tiles around it, so that an XCD's
    // tiles share a few row blocks of `a` and its L2 holds them beside all of `w`.
    // An XCD takes a stretch of the row-major tile order: a band of rows. While `w` is small that is
    // the best order: the XCD reads `w` once, and its rows of `a` are what its own workgroups of the
    // product before wrote (a prefill step's products all run over the same bands of tokens, so an
    // XCD's activations stay in its L2). With a large `w` the workgroups that run side by side on an
    // XCD, one row of tiles and all of `w`'s columns, share nothing of `w`, and every row of tiles
    // reads all of it again from memory (4,096 x 4,096 x 16,384 in 128 x 128 tiles: 3.9 GB of L2
    // misses for 0.27 GB of operands, at the memory's own speed): there the XCD's stretch goes in
    // groups of GM rows of tiles, down the rows first, so that its workgroups form a block of GM
    // rows by a few columns (half the misses; 721 -> 611 us). The bound between the two, 12 MB of
    // `w`: GPT-2 small's prefill of 2,048 tokens is 6 % slower in groups (its second feed-forward
    // product 24.2 -> 28.9 us), XL's of 8,192 tokens 6 % faster, width 4,096's 6 %.
    const int tiles_n = (N + BN - 1) / BN, tiles_m = (M + BM - 1) / BM, n_tiles = tiles_n * tiles_m;
    const int xcd = blockIdx.x % 8, base = n_tiles / 8, rem = n_tiles % 8;
    const int tile_id = xcd * base + min(xcd, rem) + blockIdx.x / 8;
    constexpr int GM = BM >= 128 ? 4 : 8;
    const bool groups = static_cast<int64_t>(N) * K > (6 << 20);
    const int per_group = groups ? GM * tiles_n : tiles_n;  // (plain rows: groups of one row of tiles)
    const int group = tile_id / per_group, first_m = group * (groups ? GM : 1), in_group = tile_id - group * per_group;
    const int gm = groups ? min(GM, tiles_m - first_m) : 1;
    m0 = (first_m + in_group % gm) * BM;
    n0 = (in_group / gm) * BN;
}

// Stores a wave's (BM / WM) x (BN / WN) sums of the tile at (m0, n0): acc[i][j] is the block of 32 x 32 (or 16 x 16: four sums a
// lane) at rows 32 i and columns 32 j of its part. `lds` may be overwritten once every wave of the workgroup has come here; it has room for what
// `staging_bytes` says.
template <int BM, int BN, int WM, int WN, int WK>
constexpr size_t staging_bytes(size_t out_bytes) {
    return out_bytes == 2 ? static_cast<size_t>(WM * WN * WK) * (BM / WM) * (BN / WN + 8) * 2 : 0;
}
template <int BM, int BN, typename OutT, int EPI, int WM, int WN, typename Sums, int TM, int TN>
__device__ __forceinline__ void store_tile(Sums (&acc)[TM][TN], bf16_t* lds, const EpiParams& epi, const PartsParams& parts, int m0, int n0, int M,
                                           int N, int vec_ok, int page_shift, int wave, int wm, int wn, int lane) {
    constexpr int BLK = sizeof(Sums) == 64 ? 32 : 16, QUADS = BLK == 32 ? 4 : 1;
    static_assert(TM * BLK * WM == BM && TN * BLK * WN == BN, "the waves' blocks are the tile");
    const int li = lane % BLK, g = lane / BLK;
    // The products were taken transposed (w's fragment as the first operand), so a lane holds one
    // row of each block, m = li, and of its columns the groups 8q + 4g + {0..3} (of 16 x 16 blocks one group): what
    // depends on the row (a token's place in the pages) is computed once, and every store is four
    // consecutive columns wide. Tiles wholly inside the output take that path without bounds
    // checks (a guarded store is a branch of its own: on an interior tile they cost as much as
    // the whole product); tiles at the bottom and the right edge take the same paths with their rows
    // and columns checked (the right edge went element by element: 7,920 x 4,800 x 1,600 in tiles
    // of 192 x 128, a column of them half outside, 144 us where 128 x 192, which fit, took 128);
    // operands that are not aligned for it go element by element.
    const bool inside = m0 + BM <= M && n0 + BN <= N, columns_inside = n0 + BN <= N;
    if constexpr (sizeof(OutT) == 2 && EPI >= 0 && EPI != kEpiResidual) {
        // bfloat16 outputs go through LDS once more (at the edges too), so that they leave as whole
        // rows: a wave lays its (BM / WM) x (BN / WN) results out row by row (bias and activation
        // applied), then every lane stores 16 bytes and eight lanes a row of 64 columns: full
        // cache lines, where the accumulators' own layout would write 16 bytes of 32 different
        // rows with every instruction (measured: 5.7 of 19.7 us on a 2,048 x 2,304 product).
        constexpr int RM = BM / WM, CN = BN / WN, LDO = CN + 8;  // padded rows, 16-byte aligned
        if (vec_ok > 1) {
            lds_barrier();  // everyone is done reading the last operand stage
            bf16_t* tile = lds + wave * RM * LDO;
            auto lay_out = [&](auto edge) {
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j) {
                        const int nb = n0 + wn * CN + j * BLK + 4 * g;
#pragma unroll
                        for (int q = 0; q < QUADS; ++q) {
                            const f32x4 b4 = epi.bias != nullptr ? *reinterpret_cast<const f32x4*>(epi.bias + (decltype(edge)::value ? min(nb + 8 * q, N - 4) : nb + 8 * q)) : f32x4{0.f, 0.f, 0.f, 0.f};
                            f32x4 v;
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                v[e] = acc[i][j][4 * q + e] + b4[e];
                                if constexpr (EPI == kEpiGeluTanh) v[e] = gelu_tanh_fast(v[e]);
                                if constexpr (EPI == kEpiGeluErf) v[e] = gelu_erf_fast(v[e]);
                            }
                            store4<bf16_t>(tile + (i * BLK + li) * LDO + j * BLK + 8 * q + 4 * g, v);
                        }
                    }
            };
            if (columns_inside) lay_out(std::false_type{});
            else lay_out(std::true_type{});
            lds_barrier();
            constexpr int CHUNKS = CN / 8, ROUNDS = RM * CHUNKS / 64;  // 16-byte pieces a row; store instructions a lane
            static_assert(RM * CHUNKS % 64 == 0, "a wave's results must be whole rounds of 64 pieces");
            const int mw = m0 + wm * RM, nw = n0 + wn * CN;
            int64_t row_base[ROUNDS];
            if constexpr (EPI == kEpiQkvPaged) {
                // the rows' places in the pages first: a load between two stores would wait for the first
#pragma unroll
                for (int t = 0; t < ROUNDS; ++t) {
                    const int slot = epi.slots[min(mw + (t * 64 + lane) / CHUNKS, M - 1)];
                    const int page = page_shift >= 0 ? slot >> page_shift : slot / epi.page_size;
                    const int off = slot - page * epi.page_size;
                    row_base[t] = static_cast<uint32_t>(slot) >= epi.num_slots ? -1 : static_cast<int64_t>(page) * epi.n_kv_head * epi.page_size * epi.hd + static_cast<int64_t>(off) * epi.hd;
                }
            }
#pragma unroll
            for (int t = 0; t < ROUNDS; ++t) {
                const int c = t * 64 + lane, row = c / CHUNKS, n = nw + (c % CHUNKS) * 8;
                if (!inside && (mw + row >= M || n >= N)) continue;  // (N is a multiple of 8: a piece is in or out)
                const u32x4 piece = *reinterpret_cast<const u32x4*>(tile + row * LDO + (c % CHUNKS) * 8);
                bf16_t* dst;
                if constexpr (EPI == kEpiQkvPaged) {
                    if (n < epi.q_dim) {
                        dst = static_cast<bf16_t*>(epi.out) + static_cast<int64_t>(mw + row) * epi.ldo + n;
                    } else {
                        if (row_base[t] < 0) continue;
                        const bool is_v = n >= epi.q_dim + epi.kv_dim;
                        const int cc = n - epi.q_dim - (is_v ? epi.kv_dim : 0);
                        const int head = cc / epi.hd, dim = cc - head * epi.hd;
                        dst = static_cast<bf16_t*>(is_v ? epi.vc : epi.kc) + row_base[t] + static_cast<int64_t>(head) * epi.page_size * epi.hd + dim;
                    }
                } else {
                    dst = static_cast<bf16_t*>(epi.out) + static_cast<int64_t>(mw + row) * epi.ldo + n;
                }
                *reinterpret_cast<u32x4*>(dst) = piece;
            }
            return;
        }
    }
    if (EPI >= 0 && vec_ok) {
        auto store = [&](auto edge) {
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const int m = m0 + wm * (BM / WM) + i * BLK + li;
                if (!inside && m >= M) continue;
                int64_t row_base = -1;
                if constexpr (EPI == kEpiQkvPaged) {
                    const int slot = epi.slots[m];
                    const int page = page_shift >= 0 ? slot >> page_shift : slot / epi.page_size;
                    const int off = slot - page * epi.page_size;
                    row_base = static_cast<uint32_t>(slot) >= epi.num_slots ? -1 : static_cast<int64_t>(page) * epi.n_kv_head * epi.page_size * epi.hd + static_cast<int64_t>(off) * epi.hd;
                }
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const int nb = n0 + wn * (BN / WN) + j * BLK + 4 * g;
                    // loads first, stores after: a load between two stores waits for the first of them
                    f32x4 b4[QUADS], r4[QUADS];
#pragma unroll
                    for (int q = 0; q < QUADS; ++q) {
                        const int n = decltype(edge)::value ? min(nb + 8 * q, N - 4) : nb + 8 * q;  // (N is a multiple of 4; columns past it: others again, not stored)
                        b4[q] = epi.bias != nullptr ? *reinterpret_cast<const f32x4*>(epi.bias + n) : f32x4{0.f, 0.f, 0.f, 0.f};
                        if constexpr (EPI == kEpiResidual)
                            r4[q] = *reinterpret_cast<const f32x4*>(epi.residual + static_cast<int64_t>(m) * epi.ldr + n);
                        if constexpr (EPI == kEpiParts) {
                            // the first part adds the rows the product is added to, their planes in order
                            r4[q] = f32x4{0.f, 0.f, 0.f, 0.f};
                            if (blockIdx.y == 0 && parts.base != nullptr) {
                                const float* bp = parts.base + static_cast<int64_t>(m) * N + n;
                                r4[q] = *reinterpret_cast<const f32x4*>(bp);
                                for (int p = 1; p < parts.n_base; ++p) r4[q] += *reinterpret_cast<const f32x4*>(bp + p * parts.base_stride);
                            }
                        }
                    }
#pragma unroll
                    for (int q = 0; q < QUADS; ++q) {
                        const int n = nb + 8 * q;
                        if (decltype(edge)::value && n >= N) continue;
                        f32x4 v;
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] = acc[i][j][4 * q + e] + b4[q][e];
                        if constexpr (EPI == kEpiResidual) {
                            *reinterpret_cast<f32x4*>(epi.residual + static_cast<int64_t>(m) * epi.ldr + n) = v + r4[q];
                        } else if constexpr (EPI == kEpiParts) {
                            float* plane = static_cast<float*>(epi.out) + blockIdx.y * parts.part_stride;
                            *reinterpret_cast<f32x4*>(plane + static_cast<int64_t>(m) * N + n) = v + r4[q];
                        } else if constexpr (EPI == kEpiQkvPaged) {
                            if (n < epi.q_dim) {
                                store4<OutT>(static_cast<OutT*>(epi.out) + static_cast<int64_t>(m) * epi.ldo + n, v);
                            } else if (row_base >= 0) {
                                const bool is_v = n >= epi.q_dim + epi.kv_dim;
                                const int c = n - epi.q_dim - (is_v ? epi.kv_dim : 0);
                                const int head = c / epi.hd, dim = c - head * epi.hd;
                                store4<OutT>(static_cast<OutT*>(is_v ? epi.vc : epi.kc) + row_base + static_cast<int64_t>(head) * epi.page_size * epi.hd + dim, v);
                            }
                        } else {
                            if constexpr (EPI == kEpiGeluTanh) {
#pragma unroll
                                for (int e = 0; e < 4; ++e) v[e] = gelu_tanh_fast(v[e]);
                            } else if constexpr (EPI == kEpiGeluErf) {
#pragma unroll
                                for (int e = 0; e < 4; ++e) v[e] = gelu_erf_fast(v[e]);
                            }
                            store4<OutT>(static_cast<OutT*>(epi.out) + static_cast<int64_t>(m) * epi.ldo + n, v);
                        }
                    }
                }
            }
        };
        if (columns_inside) store(std::false_type{});
        else store(std::true_type{});
        return;
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int m = m0 + wm * (BM / WM) + i * BLK + li;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 4 * QUADS; ++r) {
                const int n = n0 + wn * (BN / WN) + j * BLK + 8 * (r / 4) + 4 * g + r % 4;
                if constexpr (EPI == kEpiParts) {
                    if (n < N) {
                        float v = acc[i][j][r] + epilogue_bias(epi, n);
                        if (blockIdx.y == 0 && parts.base != nullptr) {
                            const float* bp = parts.base + static_cast<int64_t>(m) * N + n;
                            float b = bp[0];
                            for (int p = 1; p < parts.n_base; ++p) b += bp[p * parts.base_stride];
                            v += b;
                        }
                        (static_cast<float*>(epi.out) + blockIdx.y * parts.part_stride)[static_cast<int64_t>(m) * N + n] = v;
                    }
                } else {
                    if (n < N) epilogue_store<OutT, EPI, false>(epi, m, n, acc[i][j][r]);
                }
            }
    }
}

// How wide the stores may be (2: 16 bytes of bfloat16, 1: four outputs, 0: one), and the page size as a shift (-1: none).
template <typename OutT, int EPI>
inline void store_rules(const EpiParams& epi, int N, int& vec_ok, int& page_shift) {
    // four-wide stores need aligned rows; the cache's slots fit 32 bits (checked by the launcher)
    auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    bool vec = N % 4 == 0 && (epi.bias == nullptr || al16(epi.bias));
    page_shift = -1;
    if (EPI == kEpiResidual) {
        vec = vec && al16(epi.residual) && epi.ldr % 4 == 0;
    } else if (EPI == kEpiQkvPaged) {
        vec = vec && al16(epi.out) && al16(epi.kc) && al16(epi.vc) && epi.ldo % 4 == 0 && epi.hd % 4 == 0 && epi.q_dim % 4 == 0;
        for (int b = 0; b < 31; ++b)
            if ((1 << b) == epi.page_size) page_shift = b;
    } else {
        vec = vec && al16(epi.out) && epi.ldo % 4 == 0;
    }
    // 16-byte pieces of bfloat16 rows: row strides and the boundaries between queries, keys and
    // values in multiples of 8 elements
    bool vec16 = vec && sizeof(OutT) == 2 && N % 8 == 0;
    if (EPI == kEpiQkvPaged) vec16 = vec16 && epi.ldo % 8 == 0 && epi.hd % 8 == 0 && epi.q_dim % 8 == 0;
    else if (EPI != kEpiResidual) vec16 = vec16 && epi.ldo % 8 == 0;
    vec_ok = vec16 ? 2 : (vec ? 1 : 0);
}

// gemm_mfma_tile.hip: the tile for a product of these sizes; the product in it (2, 6: 64 x 64, three stages and four; 7, 8: 128 x 128, three and two; 21: 128 x
// 192; 9, 11: 192 x 128, two and three; 15: 256 x 256: the same bits from each); and cut over K, in tiles of 64 x 64.
int choose_gemm_tile(int M, int N, int K);
int launch_gemm_tile(int tile, const bf16_t* a, int64_t lda, const bf16_t* w, int M, int N, int K, const EpiParams& epi, hipStream_t stream);
int launch_gemm_tile_parts(const bf16_t* a, int64_t lda, const bf16_t* w, int M, int N, int K, int kparts, const EpiParams& epi, const PartsParams& parts,
                           hipStream_t stream);

// gemm_mfma_waves.hip: products of 17 to 64 rows (more are taken, row tile by row tile), whole (parts null) or cut over K.
int launch_gemm_waves(const bf16_t* a, int64_t lda, const bf16_t* w, int M, int N, int K, const EpiParams& epi, int kparts, const PartsParams* parts, hipStream_t stream);

}  // namespace liyab
