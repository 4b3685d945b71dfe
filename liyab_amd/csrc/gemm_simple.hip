// out[M,N] = a[M,K] . w[N,K]^T (+ bias) with an epilogue, for 32-bit operands
// on the matrix cores (fused multiply-adds in 32 bits: strips of 16 rows and
// tiles of 64 x 64) and for the bfloat16 shapes that the bfloat16 matrix-core
// kernels refuse, multiplied on the vector units.
//
// Both operands are contiguous along K (a row of `w` is one output feature,
// as the reference lays matrices out: include/liyab/types.h:165-184,
// y = x . W^T in include/liyab/backend.h:35). Each output element is summed
// in one fixed order that does not depend on M, so a row's result is the same
// whatever else is in the batch (include/liyab/backend.h:40-42): K in chunks
// of 64; within a chunk one chain of fused multiply-adds over ascending k that
// starts from zero; the chunks' sums added in ascending order. (Chunks, so that
// a step of few rows, which has few output elements, can still spread one
// element's sum over several waves: gemm_chunks_f32_kernel below.)
#include <type_traits>

#include "activations.h"
#include "common.h"
#include "epilogue.h"
#include "launchers.h"

namespace liyab {

constexpr int BM = 64, BN = 64, BK = 16;
constexpr int kChunk = 64;  // k of one chain of multiply-adds
static_assert(kChunk % BK == 0, "a chunk is whole tiles");

// bfloat16 operands of any size and alignment.
template <typename OutT, int EPI>
__global__ void __launch_bounds__(256)
gemm_simple_kernel(OutT* __restrict__ out, int64_t ldo, const bf16_t* __restrict__ a, int64_t lda, const bf16_t* __restrict__ w,
                   const float* __restrict__ bias, float* __restrict__ residual, int64_t ldr, int M, int N, int K) {
    __shared__ float As[BK][BM + 4];
    __shared__ float Ws[BK][BN + 4];
    const int tid = threadIdx.x;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int ty = tid / 16, tx = tid % 16;
    const int lrow = tid / 4, lk = (tid % 4) * 4;  // this thread loads 4 k of one row
    float acc[4][4] = {}, tot[4][4] = {};
    for (int k0 = 0; k0 < K; k0 += BK) {
        {
            const int m = m0 + lrow;
            const bf16_t* p = a + static_cast<int64_t>(m) * lda + k0 + lk;
#pragma unroll
            for (int i = 0; i < 4; ++i) As[lk + i][lrow] = (m < M && k0 + lk + i < K) ? to_float<bf16_t>(p[i]) : 0.0f;
            const int n = n0 + lrow;
            const bf16_t* q = w + static_cast<int64_t>(n) * K + k0 + lk;
#pragma unroll
            for (int i = 0; i < 4; ++i) Ws[lk + i][lrow] = (n < N && k0 + lk + i < K) ? to_float<bf16_t>(q[i]) : 0.0f;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < BK; ++k) {
            float av[4], wv[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) av[i] = As[k][ty * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; ++j) wv[j] = Ws[k][tx * 4 + j];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(av[i], wv[j], acc[i][j]);
        }
        if ((k0 + BK) % kChunk == 0 || k0 + BK >= K) {  // the chunk's chain ends: its sum joins the others'
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    tot[i][j] += acc[i][j];
                    acc[i][j] = 0.0f;
                }
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = m0 + ty * 4 + i;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int n = n0 + tx * 4 + j;
            if (n >= N) continue;
            float v = tot[i][j];
            if (bias != nullptr) v += bias[n];
            if constexpr (EPI == kEpiGeluTanh) v = gelu_tanh(v);
            if constexpr (EPI == kEpiGeluErf) v = gelu_erf_fast(v);
            if constexpr (EPI == kEpiResidual) {
                residual[static_cast<int64_t>(m) * ldr + n] += v;
            } else {
                out[static_cast<int64_t>(m) * ldo + n] = from_float<OutT>(v);
            }
        }
    }
}

// -- 32-bit operands ------------------------------------------------------------------------------------------
//
// The chains above on the matrix cores: v_mfma_f32_32x32x2 and _16x16x4 multiply and add in 32 bits, one
// fused multiply-add after the other over ascending k (measured on random, tiny and subnormal operands:
// 64,000 of 64,000 results have the bits of an fmaf chain; rounded once, or in another order, a third
// differ), so a chunk's chain of 64 is 32 or 16 instructions and has the bits it had on the vector units, at
// the matrix cores' 157 TFLOP/s, twice what vector multiply-adds reach that are not packed (these
// stopped at 35-57 in practice).
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(2))) float f32x2_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;

// What follows the sum (the error function in double precision).
template <int EPI>
__device__ __forceinline__ float finish_f32(float v, bool has_bias, float bias) {
    if (has_bias) v += bias;
    if constexpr (EPI == kEpiGeluTanh) v = gelu_tanh(v);
    if constexpr (EPI == kEpiGeluErf) v = gelu_erf_exact(v);
    return v;
}

// Four k of one row from a clamped address: with VEC one 16-byte load, else element by element (operands that are not
// aligned for it, a K that is no multiple of 4). What lies past K becomes zero, which adds nothing to a chain, only where the
// values go to LDS: a choice made at the load would be waited for there.
template <bool VEC>
__device__ __forceinline__ f32x4_t load4_f32(const float* __restrict__ row, int k, int K) {
    if constexpr (VEC) return *reinterpret_cast<const f32x4_t*>(row + (k < K ? k : 0));
    f32x4_t v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = row[k + i < K ? k + i : 0];
    return v;
}
__device__ __forceinline__ f32x4_t within_k(f32x4_t v, int k, int K) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = k + i < K ? v[i] : 0.0f;
    return v;
}

// Where element (m, n) of a fused query, key and value product goes: queries to rows of their own, keys and values to their
// pages (null: a token without a slot, or one outside these caches).
__device__ __forceinline__ float* qkv_place(const EpiParams& p, int m, int n) {
    if (n < p.q_dim) return static_cast<float*>(p.out) + static_cast<int64_t>(m) * p.ldo + n;
    const uint32_t slot = p.slots[m];
    if (slot >= p.num_slots) return nullptr;
    const uint32_t page = slot / static_cast<uint32_t>(p.page_size), off = slot - page * static_cast<uint32_t>(p.page_size);
    const bool is_v = n >= p.q_dim + p.kv_dim;
    const int c = n - p.q_dim - (is_v ? p.kv_dim : 0), head = c / p.hd;
    return static_cast<float*>(is_v ? p.vc : p.kc) + ((static_cast<int64_t>(page) * p.n_kv_head + head) * p.page_size + off) * p.hd + (c - head * p.hd);
}

// Many rows: tiles of 64 x 64 on four waves, a wave 32 x 32. The matrix cores set the pace (a stage of 32 k takes a compute
// unit 1,024 cycles and 16 KB of operands), so operands go through registers into one of two stages in LDS while the
// other is multiplied; they are asked for two stages ahead of their products (one stage ahead, a lone workgroup a
// compute unit waited for them: 4 x 768 x 3,072, one tile deep, 81 us against 68). An instruction takes k = 2 s from lanes 0-31
// and k = 2 s + 1 from lanes 32-63: rows lie in LDS with the even k of every eight in front of the odd ones, so that a lane
// reads its k of four instructions in 16 bytes.
// Measured, us, the 64 x 64 or 128 x 128 tiles or the row-wise kernel on vector units before: 1,222 rows, 768 -> 2,304 166 -> 50
// (87 TFLOP/s), 768 -> 3,072 192 -> 66, 3,072 -> 768 357 -> 72, 768 -> 768 103 -> 21; 4,096 rows, 768 -> 3,072 349 -> 190 (102 TFLOP/s).
// Tiles of 128 x 128 were no faster anywhere (4,096 x 3,072 x 768 192 us, 2,048 x 768 x 3,072 233 against 117), nor was a
// stage's other work strung between its products by hand.
constexpr int kTile = 64;

template <int EPI, bool VEC>
__global__ void __launch_bounds__(256)
gemm_tiled_f32_kernel(float* __restrict__ out, int64_t ldo, const float* __restrict__ a, int64_t lda, const float* __restrict__ w,
                      const float* __restrict__ bias, float* __restrict__ residual, int64_t ldr, int M, int N, int K, int vec_out, EpiParams qkv) {
    constexpr int KS = 32, LD = KS + 4;         // k a stage; padded rows: 16 lanes' 16-byte reads fall into different banks
    constexpr int STAGE = 2 * kTile * LD;       // the tile of a, then the tile of w
    __shared__ __attribute__((aligned(16))) float smem[2 * STAGE];
    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64, li = lane % 32, g = lane / 32;
    const int wm = wave / 2, wn = wave % 2;
    // an XCD takes a stretch of the tiles in groups of eight rows of tiles, down the rows first: what its L2 holds of either
    // operand is shared by the workgroups that run side by side
    const int tiles_n = (N + kTile - 1) / kTile, tiles_m = (M + kTile - 1) / kTile, n_tiles = gridDim.x;
    const int xcd = blockIdx.x % 8, tile_id = xcd * (n_tiles / 8) + min(xcd, n_tiles % 8) + blockIdx.x / 8;
    const int first = tile_id / (8 * tiles_n) * 8, within = tile_id % (8 * tiles_n), rows = min(8, tiles_m - first);
    const int m0 = (first + within % rows) * kTile, n0 = within / rows * kTile;
    const int lrow = tid / 8, lk = (tid % 8) * 4;  // this thread loads 4 k of rows lrow and lrow + 32 of either tile
    const float* src[4];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        src[i] = a + static_cast<int64_t>(min(m0 + lrow + 32 * i, M - 1)) * lda;
        src[2 + i] = w + static_cast<int64_t>(min(n0 + lrow + 32 * i, N - 1)) * K;
    }
    f32x4_t ring[2][4];
    auto fetch = [&](int k0, int stage) {
#pragma unroll
        for (int i = 0; i < 4; ++i) ring[stage][i] = load4_f32<VEC>(src[i], k0 + lk, K);
    };
    auto put = [&](int k0, int stage) {  // k = 8 q + {0, 2, 4, 6} at 8 q + 0 .. 3, the odd ones behind them
        float* s = smem + stage * STAGE + lrow * LD + (lk & ~7) + (lk & 4) / 2;
#pragma unroll
        for (int i = 0; i < 4; ++i) {  // rows lrow and lrow + 32 of a, then of w
            const f32x4_t v = within_k(ring[stage][i], k0 + lk, K);
            *reinterpret_cast<f32x2_t*>(s + 32 * i * LD) = f32x2_t{v[0], v[2]};
            *reinterpret_cast<f32x2_t*>(s + 32 * i * LD + 4) = f32x2_t{v[1], v[3]};
        }
    };
    f32x16_t acc, tot;
#pragma unroll
    for (int r = 0; r < 16; ++r) tot[r] = 0.0f;
    auto multiply = [&](int stage) {
        const float* sa = smem + stage * STAGE + (wm * 32 + li) * LD + 4 * g;
        const float* sw = smem + stage * STAGE + (kTile + wn * 32 + li) * LD + 4 * g;
        f32x4_t fa[2], fw[2];  // the next eight k are read while these multiply
        fa[0] = *reinterpret_cast<const f32x4_t*>(sa);
        fw[0] = *reinterpret_cast<const f32x4_t*>(sw);
#pragma unroll
        for (int q = 0; q < KS / 8; ++q) {
            if (q + 1 < KS / 8) {
                fa[(q + 1) & 1] = *reinterpret_cast<const f32x4_t*>(sa + (q + 1) * 8);
                fw[(q + 1) & 1] = *reinterpret_cast<const f32x4_t*>(sw + (q + 1) * 8);
            }
#pragma unroll
            for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fw[q & 1][s], fa[q & 1][s], acc, 0, 0, 0);
        }
    };
    static_assert(kChunk == 2 * KS, "a chunk is the two stages");
    const int chunks = (K + kChunk - 1) / kChunk;  // (a second stage past K is all zeros)
    fetch(0, 0);
    fetch(KS, 1);
    put(0, 0);
    fetch(2 * KS, 0);
    lds_barrier();
    for (int c = 0; c < chunks; ++c) {
        const int k0 = c * kChunk;
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
        put(k0 + KS, 1);  // (a stage's readers finished before the last barrier)
        fetch(k0 + 3 * KS, 1);
        multiply(0);
        lds_barrier();
        put(k0 + 2 * KS, 0);
        fetch(k0 + 4 * KS, 0);
        multiply(1);
        lds_barrier();
#pragma unroll
        for (int r = 0; r < 16; ++r) tot[r] += acc[r];  // the chunk's chain ends: its sum joins the others'
    }
    // w's fragment is the first operand: a lane holds one row, m, and its columns nb + 8 q + {0..3}.
    // Biases and rows to add to first: a load between two stores would wait for the first.
    const int m = m0 + wm * 32 + li, nb = n0 + wn * 32 + 4 * g;
    f32x4_t v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[q][e] = bias != nullptr ? bias[min(nb + 8 * q + e, N - 1)] : 0.0f;
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[q][e] = finish_f32<EPI>(tot[4 * q + e], bias != nullptr, v[q][e]);
    if (m >= M) return;
    if constexpr (EPI == kEpiQkvPaged) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int n = nb + 8 * q;
            if (vec_out) {  // four columns are of one head of one of the three
                float* place = n < N ? qkv_place(qkv, m, n) : nullptr;
                if (place != nullptr) *reinterpret_cast<f32x4_t*>(place) = v[q];
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float* place = n + e < N ? qkv_place(qkv, m, n + e) : nullptr;
                    if (place != nullptr) *place = v[q][e];
                }
            }
        }
        return;
    }
    float* dst = EPI == kEpiResidual ? residual + static_cast<int64_t>(m) * ldr : out + static_cast<int64_t>(m) * ldo;
    if (vec_out) {  // N is a multiple of 4: four columns are in or out together
        if constexpr (EPI == kEpiResidual) {
            f32x4_t r[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) r[q] = *reinterpret_cast<const f32x4_t*>(dst + (nb + 8 * q < N ? nb + 8 * q : 0));
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] += r[q];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (nb + 8 * q < N) *reinterpret_cast<f32x4_t*>(dst + nb + 8 * q) = v[q];
    } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int n = nb + 8 * q + e;
                if (n >= N) continue;
                if constexpr (EPI == kEpiResidual) dst[n] += v[q][e];
                else dst[n] = v[q][e];
            }
    }
}

// Few rows, or too few tiles to go round: a workgroup takes 16 rows and NB output features, its waves the chunks of K in
// turn, so that a product of few output elements still spreads over the chip. A wave brings its chunk of the rows
// of `w` and `a` through registers into LDS of its own (256 bytes a row and load, the next one or two chunks in flight
// meanwhile) and runs the chunk's chains on the matrix core, 16 x 16 x 4 an instruction; after each round of chunks the
// threads add the round's sums in chunk order. Few features a workgroup where N is small: the weights then stream
// through enough compute units (features of the block past NB repeat the last one). Reading operands from LDS set the
// pace when lanes ran the chains themselves (20 to 80 reads of 16 bytes a chunk; here 32 of 4). What bounds it is a chain: a first trip to
// memory, a round's products and sums, the epilogue's own reads, so these are asked for first of all.
// The rows may also be made here (SRC), each workgroup its own 16: the LayerNorm of 32-bit rows, or attention's splits merged, with the
// operations of layernorm.hip and of attention_decode.hip's merge, so that the bits are those of their own kernels, whose links in
// a step's chain (3.5 us each) are saved; the weights are on their way meanwhile, and the rows stay in LDS for all chunks.
constexpr int kChunkRows = 16;  // rows a workgroup
enum : int { kSrcRows = 0, kSrcNorm = 1, kSrcSplits = 2 };

// What the rows are made of where they are made here: x [M, K] and its norm, or partials [M][n_head][n_splits][hd + 4].
struct MadeRows {
    const float* x;
    const float* weight;
    const float* bias;
    float eps;
    int n_splits, n_head, hd;
};

// FORM: pieces of 4 a lane of a row (norm), splits at most (splits); not read for plain rows.
// DEPTH: chunks in flight beside the one that is multiplied. Two for one block of 16 rows, whose weights come from HBM one trip after the other; one for more rows, where the registers of two
// (104 a lane, 70 with one) and their code cost more than they hide (us, two / one: 33 rows 768 -> 3,072 9.4 / 7.9, 1,024 -> 4,096 12.3 / 10.9, 100 rows
// 15.3 / 13.9; a decode step of small's sizes, ms, 1 request 0.475 / 0.479, 8 0.540 / 0.539, 24 0.847 / 0.822, 64 1.209 / 1.172).
template <int NB, int WAVES, int EPI, bool VEC, int SRC, int FORM, int DEPTH>
__global__ void __launch_bounds__(64 * WAVES)
gemm_chunks_f32_kernel(float* __restrict__ out, int64_t ldo, const float* __restrict__ a, int64_t lda,
                       const float* __restrict__ w, const float* __restrict__ bias, float* __restrict__ residual,
                       int64_t ldr, int M_all, int N, int K, EpiParams qkv, MadeRows made) {
    const int row0 = blockIdx.y * kChunkRows, M = min(kChunkRows, M_all - row0);
    a += static_cast<int64_t>(row0) * lda;
    constexpr int LD = kChunk + 4;  // (lanes read words 4 banks apart, their neighbours in k beside them: no collisions)
    constexpr int W_LOADS = NB / 4, A_LOADS = SRC == kSrcRows ? kChunkRows / 4 : 0;  // a load covers 4 rows: 16 lanes a row, 16 bytes a lane
    static_assert(NB % 4 == 0 && NB <= 16 && kChunkRows * NB <= 64 * WAVES, "one block of features, a thread an output element");
    static_assert(SRC == kSrcRows || VEC, "rows made here are whole and aligned");
    __shared__ __attribute__((aligned(16))) float Wt[WAVES][NB][LD];
    __shared__ __attribute__((aligned(16))) float At[SRC == kSrcRows ? WAVES : 1][kChunkRows][LD];
    __shared__ float P[2][WAVES][kChunkRows][NB];  // rounds take turns, so that one barrier a round is enough
    extern __shared__ __attribute__((aligned(16))) float made_rows[];  // [M][K + 4]
    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    const int n0 = blockIdx.x * NB;
    const int chunks = (K + kChunk - 1) / kChunk, ldx = K + 4;
    const int lrow = lane / 16, lk = (lane % 16) * 4;  // as a loader
    const int li = lane % 16, g = lane / 16;           // in the matrix core's operands: row (or feature) and k
    f32x4_t wreg[DEPTH][W_LOADS], areg[DEPTH][A_LOADS + 1];
    auto fetch = [&](int c, int buf) {
        const int k = c * kChunk + lk;
#pragma unroll
        for (int i = 0; i < W_LOADS; ++i) wreg[buf][i] = load4_f32<VEC>(w + static_cast<int64_t>(min(n0 + 4 * i + lrow, N - 1)) * K, k, K);
#pragma unroll
        for (int i = 0; i < A_LOADS; ++i)
            if (4 * i < M) areg[buf][i] = load4_f32<VEC>(a + static_cast<int64_t>(min(4 * i + lrow, M - 1)) * lda, k, K);  // (the same for every lane)
    };
    float tot = 0.0f;  // of output element (tid / NB, tid % NB), for tid < 16 * NB
    float* place = nullptr;  // found while the first operands are on their way
    const int n = n0 + tid % NB, m = row0 + tid / NB;
    const bool mine = tid < kChunkRows * NB && tid / NB < M && n < N;
    float own_bias = 0.0f, own_res = 0.0f;
    auto ask = [&]() {  // the weights (and plain rows), then what the epilogue reads
        if (wave < chunks) fetch(wave, 0);
        if constexpr (DEPTH == 2)
            if (wave + WAVES < chunks) fetch(wave + WAVES, 1);
        if (mine) {
            if (bias != nullptr) own_bias = bias[n];
            if constexpr (EPI == kEpiResidual) own_res = residual[static_cast<int64_t>(m) * ldr + n];
            if constexpr (EPI == kEpiQkvPaged) place = qkv_place(qkv, m, n);
        }
    };
    if constexpr (SRC == kSrcRows) {
        ask();
    } else if constexpr (SRC == kSrcNorm) {
        const int nv = K / 4;
        const f32x4_t zero = {0.0f, 0.0f, 0.0f, 0.0f}, one = {1.0f, 1.0f, 1.0f, 1.0f};
        auto norm_row = [&](int r, auto&& between) {
            f32x4_t v[FORM], gw[FORM], gb[FORM];
#pragma unroll
            for (int j = 0; j < FORM; ++j) {
                const int at = min(lane + kWave * j, nv - 1);  // past the row: its last piece again, unused
                v[j] = reinterpret_cast<const f32x4_t*>(made.x + static_cast<int64_t>(row0 + r) * K)[at];
                gw[j] = made.weight != nullptr ? reinterpret_cast<const f32x4_t*>(made.weight)[at] : one;
                gb[j] = made.bias != nullptr ? reinterpret_cast<const f32x4_t*>(made.bias)[at] : zero;
            }
            between();
            __builtin_amdgcn_sched_barrier(0);  // the row's loads ahead of the weights': a wait for the row is then no wait for these
            float s = 0.0f;
#pragma unroll
            for (int j = 0; j < FORM; ++j)
                if (lane + kWave * j < nv) s += (v[j][0] + v[j][1]) + (v[j][2] + v[j][3]);
            const float mean = wave_sum(s) / static_cast<float>(K);
            float ss = 0.0f;
#pragma unroll
            for (int j = 0; j < FORM; ++j)
                if (lane + kWave * j < nv) {
                    const f32x4_t dev = v[j] - mean;
                    ss += (dev[0] * dev[0] + dev[1] * dev[1]) + (dev[2] * dev[2] + dev[3] * dev[3]);
                }
            const float scale = 1.0f / sqrtf(wave_sum(ss) / static_cast<float>(K) + made.eps);
#pragma unroll
            for (int j = 0; j < FORM; ++j)
                if (lane + kWave * j < nv) *reinterpret_cast<f32x4_t*>(made_rows + r * ldx + 4 * (lane + kWave * j)) = (v[j] - mean) * scale * gw[j] + gb[j];
        };
        if (wave < M) norm_row(wave, ask);
        else ask();
        for (int r = wave + WAVES; r < M; r += WAVES) norm_row(r, []() {});
        lds_barrier();  // the weights may still be on their way
    } else {
        // four consecutive k of a token a thread and item
        constexpr int ITEMS = 2;
        const int S = made.n_splits, hd4 = made.hd + 4, per = K / 4, items = M * per;
        struct Item {
            f32x4_t acc[FORM];
            f32x2_t ml[FORM];
            int place;
        } it[ITEMS];
        auto get = [&](int first) {
#pragma unroll
            for (int i = 0; i < ITEMS; ++i) {
                const int at = first + i * 64 * WAVES, ac = min(at, items - 1);  // past the end: the last one again, dropped
                const int r = ac / per, k = (ac - r * per) * 4, head = k / made.hd;
                const float* p = made.x + (static_cast<int64_t>(row0 + r) * made.n_head + head) * S * hd4;
                it[i].place = at < items ? r * ldx + k : -1;
#pragma unroll
                for (int z = 0; z < FORM; ++z) it[i].ml[z] = *reinterpret_cast<const f32x2_t*>(p + min(z, S - 1) * hd4 + made.hd);
#pragma unroll
                for (int z = 0; z < FORM; ++z) it[i].acc[z] = *reinterpret_cast<const f32x4_t*>(p + min(z, S - 1) * hd4 + k - head * made.hd);
            }
        };
        auto merge = [&]() {
#pragma unroll
            for (int i = 0; i < ITEMS; ++i) {
                float mx = -INFINITY;
#pragma unroll
                for (int z = 0; z < FORM; ++z)
                    if (z < S) mx = fmaxf(mx, it[i].ml[z][0]);
                float sum = 0.0f;
                f32x4_t o = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int z = 0; z < FORM; ++z) {
                    if (z >= S || it[i].ml[z][0] == -INFINITY) continue;
                    const float f = expf(it[i].ml[z][0] - mx);
                    sum = fmaf(f, it[i].ml[z][1], sum);
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[e] = fmaf(f, it[i].acc[z][e], o[e]);
                }
                if (it[i].place >= 0) *reinterpret_cast<f32x4_t*>(made_rows + it[i].place) = f32x4_t{o[0] / sum, o[1] / sum, o[2] / sum, o[3] / sum};
            }
        };
        get(tid);
        ask();
        __builtin_amdgcn_sched_barrier(0);
        merge();
        for (int at = tid + ITEMS * 64 * WAVES; at < items; at += ITEMS * 64 * WAVES) {
            get(at);
            merge();
        }
        lds_barrier();
    }
    const float* wl = &Wt[wave][min(li, NB - 1)][g];
    const float* al = SRC == kSrcRows ? &At[SRC == kSrcRows ? wave : 0][min(li, (M + 3) / 4 * 4 - 1)][g]  // (rows past M: some row that was written; not stored)
                                      : made_rows + min(li, M - 1) * ldx + g;
    auto round = [&](int c0, int turn, auto buffer) {
        constexpr int buf = decltype(buffer)::value;
        const int c = c0 + wave;
        if (c < chunks) {
#pragma unroll
            for (int i = 0; i < W_LOADS; ++i) *reinterpret_cast<f32x4_t*>(&Wt[wave][4 * i + lrow][lk]) = within_k(wreg[buf][i], c * kChunk + lk, K);
#pragma unroll
            for (int i = 0; i < A_LOADS; ++i)
                if (4 * i < M) *reinterpret_cast<f32x4_t*>(&At[wave][4 * i + lrow][lk]) = within_k(areg[buf][i], c * kChunk + lk, K);
            if (c + DEPTH * WAVES < chunks) fetch(c + DEPTH * WAVES, buf);
            const float* ac = SRC == kSrcRows ? al : al + c * kChunk;
            f32x4_t acc{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int k = 0; k < kChunk; k += 4) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wl[k], ac[k], acc, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r)  // a lane holds row li and the features 4 g + r
                if (4 * g + r < NB) P[turn][wave][li][4 * g + r] = acc[r];
        }
        lds_barrier();
        if (tid < kChunkRows * NB) {
            const int live = min(WAVES, chunks - c0);
            for (int v = 0; v < live; ++v) tot += P[turn][v][tid / NB][tid % NB];
        }
    };
    if constexpr (DEPTH == 2) {
        for (int c0 = 0; c0 < chunks; c0 += 2 * WAVES) {
            round(c0, 0, std::integral_constant<int, 0>{});
            if (c0 + WAVES < chunks) round(c0 + WAVES, 1, std::integral_constant<int, 1>{});
        }
    } else {
        for (int c0 = 0, turn = 0; c0 < chunks; c0 += WAVES, turn ^= 1) round(c0, turn, std::integral_constant<int, 0>{});
    }
    if (!mine) return;
    const float v = finish_f32<EPI>(tot, bias != nullptr, own_bias);
    if constexpr (EPI == kEpiResidual) residual[static_cast<int64_t>(m) * ldr + n] = own_res + v;
    else if constexpr (EPI == kEpiQkvPaged) { if (place != nullptr) *place = v; }
    else out[static_cast<int64_t>(m) * ldo + n] = v;
}

// Tiles of 64 x 64 from this many on, fewer go to the kernel by chunks, whose steady 48 TFLOP/s over 16 x 16 elements a workgroup
// beats a round of tiles that leaves compute units idle (512 rows, 3,072 -> 768, 96 tiles: 50 us against 70; 1,222 rows, 240 tiles: 116 against 72)
constexpr int kTiledMinTiles = 136;
constexpr int kFewRows = 64;  // steps of at most this many rows never take the tiles: their weights stream (64 rows, 768 -> 3,072: 8 us against 20)

template <int EPI, bool VEC>
int launch_tiled_f32(float* out, int64_t ldo, const float* a, int64_t lda, const float* w, const float* bias, float* residual, int64_t ldr, int M,
                     int N, int K, bool vec_out, const EpiParams& qkv, hipStream_t stream) {
    gemm_tiled_f32_kernel<EPI, VEC><<<((N + kTile - 1) / kTile) * ((M + kTile - 1) / kTile), 256, 0, stream>>>(out, ldo, a, lda, w, bias, residual, ldr, M, N, K, vec_out, qkv);
    return check_launch("gemm_tiled_f32");
}

template <int NB, int WAVES, int EPI, bool VEC>
int launch_chunks_f32(float* out, int64_t ldo, const float* a, int64_t lda, const float* w, const float* bias, float* residual, int64_t ldr, int M,
                      int N, int K, const EpiParams& qkv, hipStream_t stream) {
    const dim3 grid((N + NB - 1) / NB, (M + kChunkRows - 1) / kChunkRows);
    const auto kern = M <= kChunkRows ? gemm_chunks_f32_kernel<NB, WAVES, EPI, VEC, kSrcRows, 0, 2> : gemm_chunks_f32_kernel<NB, WAVES, EPI, VEC, kSrcRows, 0, 1>;
    kern<<<grid, 64 * WAVES, 0, stream>>>(out, ldo, a, lda, w, bias, residual, ldr, M, N, K, qkv, MadeRows{});
    return check_launch("gemm_chunks_f32");
}

template <int NB, int WAVES, int EPI, int SRC, int FORM>
int launch_made_as(const MadeRows& made, const float* w, int M, int N, int K, const EpiParams& epi, hipStream_t stream) {
    const size_t rows = static_cast<size_t>(M < kChunkRows ? M : kChunkRows) * (K + 4) * sizeof(float);
    constexpr size_t fixed = (WAVES * NB + kChunkRows) * (kChunk + 4) * sizeof(float) + 2 * WAVES * kChunkRows * NB * sizeof(float);
    LIYAB_REQUIRE(rows + fixed <= 160 * 1024, "gemm_made_f32: rows of %d need %zu bytes of LDS", K, rows + fixed);
    auto kern = gemm_chunks_f32_kernel<NB, WAVES, EPI, true, SRC, FORM, 2>;
    static bool ready = false;  // once per instantiation, outside any stream capture's first use
    if (!ready) {
        hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(160 * 1024 - fixed));
        ready = true;
    }
    kern<<<dim3((N + NB - 1) / NB, (M + kChunkRows - 1) / kChunkRows), 64 * WAVES, rows, stream>>>(
        static_cast<float*>(epi.out), epi.ldo, nullptr, 0, w, epi.bias, epi.residual, epi.ldr, M, N, K, epi, made);
    return check_launch("gemm_made_f32");
}
template <int EPI, int SRC, int FORM>
int launch_made(const MadeRows& made, const float* w, int M, int N, int K, const EpiParams& epi, hipStream_t stream) {
    const int64_t strips = static_cast<int64_t>(N) * ((M + kChunkRows - 1) / kChunkRows);  // (as for plain rows)
    if (strips <= 1024) return launch_made_as<4, 8, EPI, SRC, FORM>(made, w, M, N, K, epi, stream);
    if (strips <= 2048) return launch_made_as<8, 8, EPI, SRC, FORM>(made, w, M, N, K, epi, stream);
    if (strips <= 16 * 400) return launch_made_as<16, 8, EPI, SRC, FORM>(made, w, M, N, K, epi, stream);
    return launch_made_as<16, 4, EPI, SRC, FORM>(made, w, M, N, K, epi, stream);
}
template <int EPI>
int launch_norm_f32(const MadeRows& made, const float* w, int M, int N, int K, const EpiParams& epi, hipStream_t stream) {
    if (K <= 768) return launch_made<EPI, kSrcNorm, 3>(made, w, M, N, K, epi, stream);
    return launch_made<EPI, kSrcNorm, 8>(made, w, M, N, K, epi, stream);
}

template <int EPI, bool VEC>
int launch_f32_epi(float* out, int64_t ldo, const float* a, int64_t lda, const float* w, const float* bias, float* residual, int64_t ldr, int M, int N,
                   int K, const EpiParams& qkv, hipStream_t stream) {
    auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    bool vec_out = N % 4 == 0 && (EPI == kEpiResidual ? al16(residual) && ldr % 4 == 0 : al16(out) && ldo % 4 == 0);
    if (EPI == kEpiQkvPaged) vec_out = vec_out && qkv.q_dim % 4 == 0 && qkv.hd % 4 == 0 && al16(qkv.kc) && al16(qkv.vc);
#define LIYAB_ARGS out, ldo, a, lda, w, bias, residual, ldr, M, N, K
    const int64_t tiles = static_cast<int64_t>((N + 63) / 64) * ((M + 63) / 64);
    if (M > kFewRows && tiles >= kTiledMinTiles) return launch_tiled_f32<EPI, VEC>(LIYAB_ARGS, vec_out, qkv, stream);
    // Two hundred workgroups of eight waves or more: 4, 8 or 16 features each; four waves once strips of 16 features are more than
    // one and a half a compute unit (64 rows, 768 -> 3,072: 8.4 us against 12.0; 768 -> 768, 192 of them: 11.1 with eight against 14.8)
    const int64_t strips = static_cast<int64_t>(N) * ((M + kChunkRows - 1) / kChunkRows);
    if (strips <= 1024) return launch_chunks_f32<4, 8, EPI, VEC>(LIYAB_ARGS, qkv, stream);
    if (strips <= 2048) return launch_chunks_f32<8, 8, EPI, VEC>(LIYAB_ARGS, qkv, stream);
    if (strips <= 16 * 400) return launch_chunks_f32<16, 8, EPI, VEC>(LIYAB_ARGS, qkv, stream);
    return launch_chunks_f32<16, 4, EPI, VEC>(LIYAB_ARGS, qkv, stream);
#undef LIYAB_ARGS
}

template <int EPI>
int launch_f32(float* out, int64_t ldo, const float* a, int64_t lda, const float* w, const float* bias, float* residual, int64_t ldr, int M, int N,
               int K, hipStream_t stream, const EpiParams& qkv = EpiParams{}) {
    const bool vec = (reinterpret_cast<uintptr_t>(a) & 15) == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0 && lda % 4 == 0 && K % 4 == 0;
    if (vec) return launch_f32_epi<EPI, true>(out, ldo, a, lda, w, bias, residual, ldr, M, N, K, qkv, stream);
    return launch_f32_epi<EPI, false>(out, ldo, a, lda, w, bias, residual, ldr, M, N, K, qkv, stream);
}

template <typename OutT>
int launch_simple(void* out, int64_t ldo, const void* a, int64_t lda, const void* w, const float* bias,
                  float* residual, int64_t ldr, int M, int N, int K, int epi, hipStream_t stream) {
    dim3 grid((N + BN - 1) / BN, (M + BM - 1) / BM);
    auto* o = static_cast<OutT*>(out);
    auto* pa = static_cast<const bf16_t*>(a);
    auto* pw = static_cast<const bf16_t*>(w);
#define LIYAB_GO(E) \
    gemm_simple_kernel<OutT, E><<<grid, 256, 0, stream>>>(o, ldo, pa, lda, pw, bias, residual, ldr, M, N, K)
    switch (epi) {
        case kEpiNone: LIYAB_GO(kEpiNone); break;
        case kEpiGeluTanh: LIYAB_GO(kEpiGeluTanh); break;
        case kEpiGeluErf: LIYAB_GO(kEpiGeluErf); break;
        case kEpiResidual: LIYAB_GO(kEpiResidual); break;
        default: return fail(1, "gemm: unknown epilogue %d", epi);
    }
#undef LIYAB_GO
    return check_launch("gemm_simple");
}

}  // namespace liyab

using namespace liyab;

// dtype: element type of `a` and `w`; out_dtype: of `out` (ignored for the
// residual epilogue, which adds into `residual`, 32-bit, row stride ldr).
extern "C" int liyab_gemm_simple(void* out, int out_dtype, int64_t ldo, const void* a, int64_t lda, const void* w,
                                 int dtype, const float* bias, float* residual, int64_t ldr, int M, int N, int K,
                                 int epi, hipStream_t stream) {
    LIYAB_REQUIRE(a && w, "gemm: null operand");
    LIYAB_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm: bad sizes M=%d N=%d K=%d", M, N, K);
    LIYAB_REQUIRE(lda >= K, "gemm: lda %lld < K %d", static_cast<long long>(lda), K);
    if (epi == kEpiResidual) {
        LIYAB_REQUIRE(residual != nullptr && ldr >= N, "gemm: the residual epilogue needs a residual of row stride >= N");
    } else {
        LIYAB_REQUIRE(out != nullptr && ldo >= N, "gemm: needs an output of row stride >= N");
    }
    if (M == 0) return 0;
    if (dtype == kF32) {
        LIYAB_REQUIRE(epi == kEpiResidual || out_dtype == kF32, "gemm: 32-bit operands give a 32-bit output");
        auto* o = static_cast<float*>(out);
        auto *pa = static_cast<const float*>(a), *pw = static_cast<const float*>(w);
        switch (epi) {
            case kEpiNone: return launch_f32<kEpiNone>(o, ldo, pa, lda, pw, bias, residual, ldr, M, N, K, stream);
            case kEpiGeluTanh: return launch_f32<kEpiGeluTanh>(o, ldo, pa, lda, pw, bias, residual, ldr, M, N, K, stream);
            case kEpiGeluErf: return launch_f32<kEpiGeluErf>(o, ldo, pa, lda, pw, bias, residual, ldr, M, N, K, stream);
            case kEpiResidual: return launch_f32<kEpiResidual>(o, ldo, pa, lda, pw, bias, residual, ldr, M, N, K, stream);
            default: return fail(1, "gemm: unknown epilogue %d", epi);
        }
    }
    if (dtype == kBF16) {
        if (out_dtype == kF32) return launch_simple<float>(out, ldo, a, lda, w, bias, residual, ldr, M, N, K, epi, stream);
        if (out_dtype == kBF16) return launch_simple<bf16_t>(out, ldo, a, lda, w, bias, residual, ldr, M, N, K, epi, stream);
        return fail(1, "gemm: unknown output dtype %d", out_dtype);
    }
    return fail(1, "gemm: unknown dtype %d", dtype);
}

// The fused query, key and value product of the 32-bit path: queries to epi->out, keys and values into their pages (epi->mode:
// the paged one). The bits are liyab_gemm_simple's followed by liyab_kv_write's, without that launch and its trip through memory (4.6 us
// a layer of a decode step).
extern "C" int liyab_gemm_f32_qkv(const float* a, int64_t lda, const float* w, int M, int N, int K, const EpiParams* epi, hipStream_t stream) {
    LIYAB_REQUIRE(a && w && epi, "gemm_f32_qkv: null operand");
    LIYAB_REQUIRE(M >= 0 && N > 0 && K > 0 && lda >= K, "gemm_f32_qkv: bad sizes M=%d N=%d K=%d lda=%lld", M, N, K, static_cast<long long>(lda));
    LIYAB_REQUIRE(epi->mode == kEpiQkvPaged && epi->out_dtype == kF32, "gemm_f32_qkv: takes the paged epilogue with 32-bit caches only");
    if (int rc = check_epilogue(*epi, M, N)) return rc;
    if (M == 0) return 0;
    return launch_f32<kEpiQkvPaged>(static_cast<float*>(epi->out), epi->ldo, a, lda, w, epi->bias, nullptr, 0, M, N, K, stream, *epi);
}

// The same products over rows that the kernel makes itself (K a multiple of 64, operands 16-byte aligned): LayerNorm(x) of 32-bit rows x [M, K],
// K <= 2048, every epilogue but the residual one; or attention's splits [M][n_head][n_splits <= 8][hd + 4] merged, K = n_head * hd, the residual
// epilogue. As many rows as a workgroup's LDS holds beside its chunks (16 of up to 1,664 whatever N; of 2,048 up to 13): more is refused. The bits are those of
// liyab_layernorm or liyab_attention_merge followed by the product.
static int check_made(const void* x, const void* w, int M, int N, int K, const EpiParams* epi) {
    auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    LIYAB_REQUIRE(x && w && epi, "gemm_made_f32: null operand");
    LIYAB_REQUIRE(M >= 0 && N > 0 && K > 0 && K % kChunk == 0, "gemm_made_f32: bad sizes M=%d N=%d K=%d (a multiple of 64)", M, N, K);
    LIYAB_REQUIRE(al16(x) && al16(w), "gemm_made_f32: operands must be 16-byte aligned");
    LIYAB_REQUIRE(epi->mode == kEpiResidual || epi->out_dtype == kF32, "gemm_made_f32: 32-bit operands give a 32-bit output");
    return check_epilogue(*epi, M, N);
}
extern "C" int liyab_gemm_f32_ln(const float* x, const float* ln_weight, const float* ln_bias, float eps, const float* w, int M, int N, int K,
                                 const EpiParams* epi, hipStream_t stream) {
    if (int rc = check_made(x, w, M, N, K, epi)) return rc;
    LIYAB_REQUIRE(K <= 2048 && eps >= 0.0f, "gemm_f32_ln: rows of %d (at most 2048), eps %g", K, static_cast<double>(eps));
    LIYAB_REQUIRE(((reinterpret_cast<uintptr_t>(ln_weight) | reinterpret_cast<uintptr_t>(ln_bias)) & 15) == 0, "gemm_f32_ln: operands must be 16-byte aligned");
    if (M == 0) return 0;
    const MadeRows made{x, ln_weight, ln_bias, eps, 0, 0, 0};
    switch (epi->mode) {
        case kEpiNone: return launch_norm_f32<kEpiNone>(made, w, M, N, K, *epi, stream);
        case kEpiGeluTanh: return launch_norm_f32<kEpiGeluTanh>(made, w, M, N, K, *epi, stream);
        case kEpiGeluErf: return launch_norm_f32<kEpiGeluErf>(made, w, M, N, K, *epi, stream);
        case kEpiQkvPaged: return launch_norm_f32<kEpiQkvPaged>(made, w, M, N, K, *epi, stream);
        default: return fail(1, "gemm_f32_ln: epilogue %d is not taken", epi->mode);
    }
}
extern "C" int liyab_gemm_f32_splits(const float* partials, int n_splits, int n_head, int hd, const float* w, int M, int N, const EpiParams* epi,
                                     hipStream_t stream) {
    LIYAB_REQUIRE(n_splits >= 1 && n_splits <= 8 && n_head > 0 && hd > 0 && hd % 4 == 0 && static_cast<int64_t>(n_head) * hd <= 8192,
                  "gemm_f32_splits: %d splits (1 to 8) of %d heads of %d", n_splits, n_head, hd);
    const int K = n_head * hd;
    if (int rc = check_made(partials, w, M, N, K, epi)) return rc;
    LIYAB_REQUIRE(epi->mode == kEpiResidual, "gemm_f32_splits: takes the residual epilogue");
    if (M == 0) return 0;
    const MadeRows made{partials, nullptr, nullptr, 0.0f, n_splits, n_head, hd};
    if (n_splits <= 4) return launch_made<kEpiResidual, kSrcSplits, 4>(made, w, M, N, K, *epi, stream);
    return launch_made<kEpiResidual, kSrcSplits, 8>(made, w, M, N, K, *epi, stream);
}
