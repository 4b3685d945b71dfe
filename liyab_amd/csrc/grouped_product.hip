// Many small products with one launch: out rows of group g = a rows . w[g]^T, where a group is a
// head (every row of the step, its own columns of `a` and of `out`) or an expert (the rows that a
// router sent to it, listed in tiles of kGroupedRows places by liyab_moe_align).
//
//   idx   = the row's number: m for heads; rows_list[place] for listed rows (-1: an empty place)
//   a row = a + (idx / a_div) * lda + g * a_group_cols       (a_div: entries a token, so that a
//                                                             token's row serves each of its experts)
//   w[g]  = w + g * N * K, a row an output feature ([N, K], K contiguous)
//   out   = out + (idx + (idx / out_div) * out_extra) * ldo + g * out_group_cols + column
//   value = acc0, or relu(acc0)^2 with act = 1   (one matrix)
//         = silu(acc0) * acc1                    (two matrices: a gated unit's first products)
//         = g sigmoid(slope g) (u + shift), g = min(acc0, limit), u = clamp(acc1, -limit, limit), with act = 2 (two matrices, clamped)
//     then * row_scale[idx] (a router's weight), * sigmoid(gate[idx * gate_stride + g * N + column])
//     (the gate's logits float32 or bfloat16)
//
// bfloat16 operands with K a multiple of 8 run on the matrix cores in tiles of 64 rows (K a multiple of 64: 64 or 128 rows of weights,
// grouped_tile_kernel; other K: 64 x 64, four waves of 32 x 32, through registers; both with 32-bit sums in one order); float32 operands, and sizes the matrix
// kernel does not take, run as plain multiply-adds in 32-bit (tiles of 64 x 64, a thread 4 x 4).
// Every output element is a sum over k in one order whatever rows share its tile.
#include "common.h"
#include "launchers.h"
#include "ring.h"

namespace liyab {

constexpr int kGroupedRows = 64;  // rows a tile; liyab_moe_align lays its lists out in these,
constexpr int kSkinnyRows = 16;   // or in these for steps whose experts get few rows each

struct GroupedParams {
    const void* a;
    int64_t lda;
    int a_div, a_group_cols;
    const void* w0;
    const void* w1;
    void* out;
    int64_t ldo;
    int out_group_cols, out_dtype;
    const int* rows_list;   // null: rows 0..M-1 and the group is blockIdx.z
    const int* tile_group;  // with rows_list: the group of each tile of rows, -1 for a tile nobody uses
    const float* row_scale;
    const void* gate;  // logits of a gate on the output, float32 or bfloat16 (gate_dtype), or null
    int64_t gate_stride;
    int gate_dtype;
    int M, N, K;
    int block;  // places a tile of rows_list: kGroupedRows, or kSkinnyRows for steps of few rows
    int act;        // one matrix: 0 = the sums as they are, 1 = the square of their positive part (relu(.)^2); two: 0 = silu(u) v, 2 = clamped
    int out_div, out_extra;  // `out_extra` rows of `out` are left free behind each `out_div` rows (a token's entries), for results another product adds
    float limit, slope, shift;  // act = 2
};

__device__ __forceinline__ float gp_sigmoid(float z) { return 1.0f / (1.0f + expf(-z)); }

// The output of row `idx`, feature n of group g, from the sums of the one or two matrices.
template <int NW>
__device__ __forceinline__ float grouped_act(const GroupedParams& p, float v0, float v1) {
    float v = v0;
    if constexpr (NW == 2) {
        if (p.act == 2) {
            const float g = fminf(v0, p.limit), u = fminf(fmaxf(v1, -p.limit), p.limit);
            v = g * gp_sigmoid(p.slope * g) * (u + p.shift);
        } else v = v0 * gp_sigmoid(v0) * v1;
    }
    else if (p.act == 1) v = v0 > 0.0f ? v0 * v0 : 0.0f;
    return v;
}
template <int NW>
__device__ __forceinline__ float grouped_value(const GroupedParams& p, int idx, int g, int n, float v0, float v1) {
    float v = grouped_act<NW>(p, v0, v1);
    if (p.row_scale != nullptr) v *= p.row_scale[idx];
    if (p.gate != nullptr) {
        const int64_t ga = static_cast<int64_t>(idx) * p.gate_stride + static_cast<int64_t>(g) * p.N + n;
        v *= gp_sigmoid(p.gate_dtype == kF32 ? static_cast<const float*>(p.gate)[ga] : bf16_to_float(static_cast<const bf16_t*>(p.gate)[ga]));
    }
    return v;
}

// Where row `idx` of group g begins in `out`.
__device__ __forceinline__ int64_t grouped_place(const GroupedParams& p, int idx, int g) {
    return static_cast<int64_t>(idx + (idx / p.out_div) * p.out_extra) * p.ldo + static_cast<int64_t>(g) * p.out_group_cols;
}

template <int NW>
__device__ __forceinline__ void grouped_store(const GroupedParams& p, int idx, int g, int n, float v0, float v1) {
    const float v = grouped_value<NW>(p, idx, g, n, v0, v1);
    const int64_t at = grouped_place(p, idx, g) + n;
    if (p.out_dtype == kF32)
        static_cast<float*>(p.out)[at] = v;
    else
        static_cast<bf16_t*>(p.out)[at] = float_to_bf16(v);
}

// The rows of this workgroup's tile: their numbers into `idx` (LDS, kGroupedRows ints), the group returned (-1: nothing to do).
__device__ __forceinline__ int grouped_rows(const GroupedParams& p, int* idx) {
    const int tile = blockIdx.x;
    int g;
    if (p.rows_list != nullptr) {
        g = p.tile_group[tile];
        if (g < 0) return -1;
        for (int i = threadIdx.x; i < kGroupedRows; i += blockDim.x) idx[i] = i < p.block ? p.rows_list[tile * p.block + i] : -1;
    } else {
        g = blockIdx.z;
        for (int i = threadIdx.x; i < kGroupedRows; i += blockDim.x) {
            const int m = tile * kGroupedRows + i;
            idx[i] = m < p.M ? m : -1;
        }
    }
    __syncthreads();
    return g;
}

typedef __attribute__((ext_vector_type(8))) __bf16 gp_bf16x8;
typedef __attribute__((ext_vector_type(16))) float gp_floatx16;
typedef __attribute__((ext_vector_type(4))) uint32_t gp_u32x4;

constexpr int GPK = 64;       // k per LDS tile
constexpr int GPLD = GPK + 8;  // padded row, in elements

template <int NW>
__global__ void __launch_bounds__(256)
grouped_mfma_kernel(GroupedParams p) {
    __shared__ __attribute__((aligned(16))) bf16_t lds[(1 + NW) * 64 * GPLD];
    __shared__ int idx[kGroupedRows];
    const int g = grouped_rows(p, idx);
    if (g < 0) return;
    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    const int wm = wave / 2, wn = wave % 2;
    const int n0 = blockIdx.y * 64;
    const int li = lane % 32, lk = (lane / 32) * 8;
    const int N = p.N, K = p.K;
    const bf16_t* a = static_cast<const bf16_t*>(p.a) + static_cast<int64_t>(g) * p.a_group_cols;
    const bf16_t* w[2] = {static_cast<const bf16_t*>(p.w0) + static_cast<int64_t>(g) * N * K,
                          NW == 2 ? static_cast<const bf16_t*>(p.w1) + static_cast<int64_t>(g) * N * K : nullptr};
    gp_floatx16 acc[NW];
#pragma unroll
    for (int u = 0; u < NW; ++u)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[u][r] = 0.0f;

    // a thread's two 16-byte pieces of each operand tile: rows tid / 8 and tid / 8 + 32, k piece tid % 8.
    // Every load is made, from a row that exists (an empty place reads the first row, a feature past N the
    // first feature, a piece past K the row's last piece) and masked afterwards: a load under a branch is
    // waited for where the branch ends, and the pieces of kStages tiles of K are to be in flight together.
    const int row_a = tid / 8, kc = (tid % 8) * 8;
    const bf16_t* a_src[2];
    const bf16_t* w_src[NW][2];
    bool a_ok[2], w_ok[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int id = idx[row_a + 32 * i];
        a_ok[i] = id >= 0;
        a_src[i] = a + static_cast<int64_t>(a_ok[i] ? id / p.a_div : 0) * p.lda;
        const int n = n0 + row_a + 32 * i;
        w_ok[i] = n < N;
#pragma unroll
        for (int u = 0; u < NW; ++u) w_src[u][i] = w[u] + static_cast<int64_t>(w_ok[i] ? n : 0) * K;
    }
    const gp_u32x4 zero = {0, 0, 0, 0};
    constexpr int kStages = NW == 2 ? 1 : 2;  // tiles of K whose pieces are in flight: a tile's trip from memory is most of its time otherwise
    gp_u32x4 ra[kStages][2], rw[kStages][NW][2];
    auto fetch = [&](int s, int k0) {
        const int k = min(k0 + kc, K - 8);
        const bool in_k = k0 + kc < K;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const gp_u32x4 va = *reinterpret_cast<const gp_u32x4*>(a_src[i] + k);
            ra[s][i] = (a_ok[i] && in_k) ? va : zero;
#pragma unroll
            for (int u = 0; u < NW; ++u) {
                const gp_u32x4 vw = *reinterpret_cast<const gp_u32x4*>(w_src[u][i] + k);
                rw[s][u][i] = (w_ok[i] && in_k) ? vw : zero;
            }
        }
    };
    const int nk = (K + GPK - 1) / GPK;
#pragma unroll
    for (int s = 0; s < kStages; ++s) fetch(s, min(s, nk - 1) * GPK);  // (a stage past the last tile reads the last one again, unused)
    for (int kb = 0; kb < nk; kb += kStages) {
#pragma unroll
        for (int s = 0; s < kStages; ++s) {
            if (kb + s < nk) {  // (the same for every thread of the workgroup)
                lds_barrier();  // the previous tile's fragments have been read
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    *reinterpret_cast<gp_u32x4*>(lds + (row_a + 32 * i) * GPLD + kc) = ra[s][i];
#pragma unroll
                    for (int u = 0; u < NW; ++u) *reinterpret_cast<gp_u32x4*>(lds + ((1 + u) * 64 + row_a + 32 * i) * GPLD + kc) = rw[s][u][i];
                }
                fetch(s, min(kb + s + kStages, nk - 1) * GPK);
                lds_barrier();
                const bf16_t* Ab = lds + (wm * 32 + li) * GPLD + lk;
#pragma unroll
                for (int ks = 0; ks < GPK; ks += 16) {
                    const gp_bf16x8 fa = *reinterpret_cast<const gp_bf16x8*>(Ab + ks);
#pragma unroll
                    for (int u = 0; u < NW; ++u) {
                        const gp_bf16x8 fw = *reinterpret_cast<const gp_bf16x8*>(lds + ((1 + u) * 64 + wn * 32 + li) * GPLD + lk + ks);
                        acc[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa, fw, acc[u], 0, 0, 0);
                    }
                }
            }
        }
    }
    // C block layout: a lane holds column li; rows 8 * (r / 4) + 4 * (lane / 32) + r % 4
    const int n = n0 + wn * 32 + li;
    if (n >= N) return;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int id = idx[wm * 32 + 4 * (lane / 32) + 8 * (r / 4) + r % 4];
        if (id >= 0) grouped_store<NW>(p, id, g, n, acc[0][r], NW == 2 ? acc[NW - 1][r] : 0.0f);
    }
}

// The same for K a multiple of 64: 64 rows by 128 rows of weights (128 features of one matrix, or 64 of each of two) in blocks of 16 x 16,
// operands straight from global memory into a ring of stages in LDS as in gemm_mfma_tile.hip, the rows of `a` from wherever the list says.
// What bounds it: the operands, at what a compute unit takes in (24 KiB a stage of 64 k for 1 MFLOP), and with them which L2 they come
// from. A group's rows stand side by side in the list, so an XCD takes a stretch of the tiles in use: its rows of `a` and a column of
// weights at a time, for all of its tiles in turn, stay in its L2, where tiles dealt out over the XCDs had every one of them read every expert's weights.
// The gates' logits and a row's scale and place are asked for before the walk: a load under a choice in the epilogue is waited for there (the first
// of the products below took 41 us so). us before (the kernel above) and now, the same bits: 3,280 entries of 8 experts, 768 -> 2 x 1,536 54 -> 33, 1,536 -> 768
// 32 -> 21, 768 -> 2 x 768 30 -> 17.2; 10,000 entries 102 -> 83 and 87 -> 45; heads, 1,640 rows of 12, 128 -> 64 with a gate 10.5 -> 6.8, 64 -> 128 8.3 -> 5.5.
typedef __attribute__((ext_vector_type(4))) float gp_f32x4;

// WR: rows of weights a tile, WR / NW features of each matrix.
template <int NW, int WR, int STAGES>
__global__ void __launch_bounds__(256, 2)
grouped_tile_kernel(GroupedParams p, int n_tiles, int n_groups, int vec_ok, int gate_vec) {
    constexpr int BN = WR / NW, TN = WR / 32, STAGE = (kGroupedRows + WR) * GPK;  // features a tile, a wave's blocks of them, elements a stage
    constexpr int A_LOADS = 2, W_LOADS = WR / 32, LOADS = A_LOADS + W_LOADS;      // a wave's loads a stage, 1 KiB each: 8 rows of 64 k
    extern __shared__ __attribute__((aligned(1024))) bf16_t ring[];
    __shared__ int idx[kGroupedRows];
    __shared__ int64_t places[kGroupedRows];  // where a row begins in `out`
    __shared__ float scales[kGroupedRows];
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64), wm = wave / 2, wn = wave % 2;
    const int N = p.N, K = p.K, columns = (N + BN - 1) / BN;

    // the tiles in use (up to the last that has a group), then this workgroup's. A list's spare tiles are no more than its experts, so that a look at the
    // last 256 tells, and beyond it they all count as used (every workgroup looking at every tile was the larger part of a long list's time: 400,000 entries
    // of 64 experts, 256 -> 2 x 128 233 us so, 161 now; 100,000 of 8, 768 -> 768 291 and 275).
    __shared__ int last;
    if (p.rows_list != nullptr) {
        if (tid == 0) last = max(n_tiles - 256, 0);
        __syncthreads();
        const int t = n_tiles - 256 + tid;
        if (t >= 0 && p.tile_group[t] >= 0) atomicMax(&last, t + 1);
        __syncthreads();
    }
    const int used = p.rows_list != nullptr ? last : n_tiles;
    const int per_group = used * columns, total = per_group * n_groups;  // (n_groups: heads; 1 with a list)
    const int xcd = blockIdx.x % 8, base = total / 8, rem = total % 8, slot = blockIdx.x / 8;
    if (slot >= base + (xcd < rem ? 1 : 0)) return;
    const int id = xcd * base + min(xcd, rem) + slot, in_group = id % per_group;
    const int stretch = (used + 7) / 8;  // tiles whose columns are taken in turn
    const int block = in_group / (stretch * columns), first = block * stretch, here = min(stretch, used - first), rest = in_group - first * columns;
    const int tile = first + rest % here, n0 = rest / here * BN;
    const int g = p.rows_list != nullptr ? p.tile_group[tile] : id / per_group;
    if (g < 0) return;
    if (tid < kGroupedRows) {
        const int place = tile * kGroupedRows + tid;
        const int id_row = p.rows_list != nullptr ? p.rows_list[place] : place < p.M ? place : -1;
        idx[tid] = id_row;
        places[tid] = grouped_place(p, max(id_row, 0), g);
        if (p.row_scale != nullptr) scales[tid] = p.row_scale[max(id_row, 0)];
    }
    __syncthreads();
    const int li = lane % 16, q = lane / 16;
    // the gates' logits are asked for first: they are here when the sums are
    gp_f32x4 gates[2][TN];
    if (NW == 1 && p.gate != nullptr) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int64_t at = static_cast<int64_t>(max(idx[wm * 32 + i * 16 + li], 0)) * p.gate_stride + static_cast<int64_t>(g) * N;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int n = n0 + wn * (BN / 2) + j * 16 + 4 * q;
                if (gate_vec) {
                    const int64_t from = at + min(n, N - 4);
                    if (p.gate_dtype == kF32) gates[i][j] = *reinterpret_cast<const gp_f32x4*>(static_cast<const float*>(p.gate) + from);
                    else {
                        const uint2 b = *reinterpret_cast<const uint2*>(static_cast<const bf16_t*>(p.gate) + from);
                        gates[i][j] = gp_f32x4{__uint_as_float(b.x << 16), __uint_as_float(b.x & 0xffff0000u), __uint_as_float(b.y << 16), __uint_as_float(b.y & 0xffff0000u)};
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int64_t from = at + min(n + e, N - 1);
                        gates[i][j][e] = p.gate_dtype == kF32 ? static_cast<const float*>(p.gate)[from] : bf16_to_float(static_cast<const bf16_t*>(p.gate)[from]);
                    }
                }
            }
        }
    }

    // Piece c of a row lies at c ^ ((row / 2) % 8): 16 consecutive rows at one piece fall on different banks. An empty place reads the first
    // row, a feature past N the last one: computed, never stored.
    const bf16_t* src[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int row = (i < A_LOADS ? wave * A_LOADS + i : wave * W_LOADS + i - A_LOADS) * 8 + lane / 8;
        const int c = ((lane % 8) ^ ((row >> 1) & 7)) * 8;
        if (i < A_LOADS) {
            src[i] = static_cast<const bf16_t*>(p.a) + static_cast<int64_t>(max(idx[row], 0) / p.a_div) * p.lda + static_cast<int64_t>(g) * p.a_group_cols + c;
        } else {
            const void* w = NW == 2 && row >= BN ? p.w1 : p.w0;
            src[i] = static_cast<const bf16_t*>(w) + (static_cast<int64_t>(g) * N + min(n0 + row % BN, N - 1)) * K + c;
        }
    }
    auto issue = [&](int begin, int end, int unit, int stage) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            if (i < begin || i >= end) continue;
            bf16_t* to = ring + stage * STAGE + (i < A_LOADS ? wave * A_LOADS + i : 8 + wave * W_LOADS + i - A_LOADS) * 512;
            const bf16_t* from = src[i] + unit * GPK;
            __builtin_amdgcn_global_load_lds(from, (lds_void_ptr)(to), 16, 0, 0);
        }
    };
    // a wave's 32 rows by 64 rows of weights, 32 features of each matrix where there are two: acc[i][j]
    gp_f32x4 acc[2][TN];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = gp_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const int swizzle = (li >> 1) & 7;
    auto multiply = [&](int stage, int half) {  // 32 k
        const bf16_t* piece = ring + stage * STAGE + ((4 * half + q) ^ swizzle) * 8 + li * GPK;
        gp_bf16x8 fa[2], fw[TN];
#pragma unroll
        for (int j = 0; j < TN; ++j) fw[j] = *reinterpret_cast<const gp_bf16x8*>(piece + (kGroupedRows + (NW == 2 ? (j / 2) * BN + wn * 32 + (j % 2) * 16 : wn * (BN / 2) + j * 16)) * GPK);
#pragma unroll
        for (int i = 0; i < 2; ++i) fa[i] = *reinterpret_cast<const gp_bf16x8*>(piece + (wm * 32 + i * 16) * GPK);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[j], fa[i], acc[i][j], 0, 0, 0);
    };
    const int units = K / GPK;
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s)
        if (s < units) issue(0, LOADS, s, s);
    for (int u = 0, stage = 0, next = STAGES - 1; u < units; ++u) {
        // unit u must have landed; the loads of the unit after it may be in flight (a wave's loads complete in order)
        if (STAGES > 2 && u + 1 < units) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(STAGES > 2 ? LOADS : 0) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        // everyone's loads of unit u are in LDS, everyone is done reading unit u - 1: its stage takes unit u + 2
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        const bool more = u + STAGES - 1 < units;
        if (more) issue(0, LOADS / 2, u + STAGES - 1, next);
        multiply(stage, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (more) issue(LOADS / 2, LOADS, u + STAGES - 1, next);
        multiply(stage, 1);
        __builtin_amdgcn_sched_barrier(0);
        stage = stage + 1 == STAGES ? 0 : stage + 1;
        next = next + 1 == STAGES ? 0 : next + 1;
    }
    // a lane holds row li of a block and its features 4 q .. 4 q + 3: through LDS, so that rows leave whole
    constexpr int LDO = BN + 4;  // floats
    float* const results = reinterpret_cast<float*>(ring);
    lds_barrier();  // everyone is done with the last stage
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int row = wm * 32 + i * 16 + li;
#pragma unroll
        for (int j = 0; j < TN / NW; ++j) {
            const int at = wn * (BN / 2) + j * 16 + 4 * q;
            gp_f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = grouped_act<NW>(p, acc[i][j][e], NW == 2 ? acc[i][j + TN - TN / NW][e] : 0.0f);
                if (p.row_scale != nullptr) v[e] *= scales[row];
                if (NW == 1 && p.gate != nullptr) v[e] *= gp_sigmoid(gates[i][j][e]);
            }
            *reinterpret_cast<gp_f32x4*>(results + row * LDO + at) = v;
        }
    }
    lds_barrier();
    if (vec_ok) {  // N, strides and the groups' columns are multiples of 8, `out` is aligned: eight features at a time
        for (int c = tid; c < kGroupedRows * BN / 8; c += 256) {
            const int row = c / (BN / 8), n = c % (BN / 8) * 8, id_row = idx[row];
            if (id_row < 0 || n0 + n >= N) continue;
            const gp_f32x4 lo = *reinterpret_cast<const gp_f32x4*>(results + row * LDO + n), hi = *reinterpret_cast<const gp_f32x4*>(results + row * LDO + n + 4);
            const int64_t at = places[row] + n0 + n;
            if (p.out_dtype == kF32) {
                *reinterpret_cast<gp_f32x4*>(static_cast<float*>(p.out) + at) = lo;
                *reinterpret_cast<gp_f32x4*>(static_cast<float*>(p.out) + at + 4) = hi;
            } else {
                gp_bf16x8 b;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    b[e] = static_cast<__bf16>(lo[e]);
                    b[4 + e] = static_cast<__bf16>(hi[e]);
                }
                *reinterpret_cast<gp_bf16x8*>(static_cast<bf16_t*>(p.out) + at) = b;
            }
        }
    } else {
        for (int c = tid; c < kGroupedRows * BN; c += 256) {
            const int row = c / BN, n = c % BN, id_row = idx[row];
            if (id_row < 0 || n0 + n >= N) continue;
            const int64_t at = places[row] + n0 + n;
            const float v = results[row * LDO + n];
            if (p.out_dtype == kF32) static_cast<float*>(p.out)[at] = v;
            else static_cast<bf16_t*>(p.out)[at] = float_to_bf16(v);
        }
    }
}

template <int NW, int WR, int STAGES>
int launch_grouped_tile(const GroupedParams& p, int n_tiles, int n_groups, hipStream_t stream) {
    constexpr int smem = STAGES * (kGroupedRows + WR) * GPK * 2, BN = WR / NW;
    static_assert(smem >= kGroupedRows * (BN + 4) * 4, "the results fit where the stages were");
    static bool ready = false;  // once per instantiation, outside any stream capture's first use
    if (!ready) {
        hipFuncSetAttribute(reinterpret_cast<const void*>(grouped_tile_kernel<NW, WR, STAGES>), hipFuncAttributeMaxDynamicSharedMemorySize, smem);
        ready = true;
    }
    const bool vec = p.N % 8 == 0 && p.ldo % 8 == 0 && p.out_group_cols % 8 == 0 && (reinterpret_cast<uintptr_t>(p.out) & 15) == 0;
    const size_t gate_elt = p.gate_dtype == kF32 ? 16 : 8;
    const bool gate_vec = p.N % 4 == 0 && p.gate_stride % 4 == 0 && reinterpret_cast<uintptr_t>(p.gate) % gate_elt == 0;
    grouped_tile_kernel<NW, WR, STAGES><<<n_tiles * ((p.N + BN - 1) / BN) * n_groups, 256, smem, stream>>>(p, n_tiles, n_groups, vec, gate_vec);
    return check_launch("grouped_product");
}

// Few rows a group (decoding: an expert gets a token or two): the product is a stream of the group's
// weights, and what matters is how many workgroups pull on it. A workgroup owns 16 output features and one
// tile of 16 row places; its four waves deal the units of 64 k among themselves and add their sums through
// LDS in wave order. With v_mfma_f32_16x16x32_bf16 the weights are the first operand and the rows the second,
// both straight from global memory into registers, 16 bytes a lane, a trip ahead of the multiplies. The order
// of an element's sum depends on K alone.
typedef __attribute__((ext_vector_type(4))) float gp_floatx4;
union GpFrag {
    gp_u32x4 u;
    gp_bf16x8 v;
};

template <int NW>
__global__ void __launch_bounds__(256)
grouped_skinny_kernel(GroupedParams p) {
    __shared__ float red[4 * NW * 256];
    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    const int i = lane % 16, q = lane / 16;
    const int tile = blockIdx.x;
    int g;
    if (p.rows_list != nullptr) {
        g = p.tile_group[tile];
        if (g < 0) return;
    } else {
        g = blockIdx.z;
    }
    auto row_id = [&](int place) {
        if (p.rows_list != nullptr) return p.rows_list[tile * kSkinnyRows + place];
        const int m = tile * kSkinnyRows + place;
        return m < p.M ? m : -1;
    };
    const int N = p.N, K = p.K, n0 = blockIdx.y * 16;
    const int my_id = row_id(i);
    // an empty place reads the first row, a feature past N the last one: computed, never stored
    const bf16_t* arow = static_cast<const bf16_t*>(p.a) + static_cast<int64_t>(my_id >= 0 ? my_id / p.a_div : 0) * p.lda + static_cast<int64_t>(g) * p.a_group_cols;
    const int64_t wrow = (static_cast<int64_t>(g) * N + min(n0 + i, N - 1)) * K;
    const bf16_t* w[2] = {static_cast<const bf16_t*>(p.w0) + wrow, NW == 2 ? static_cast<const bf16_t*>(p.w1) + wrow : nullptr};
    const gp_u32x4 zero = {0, 0, 0, 0};
    // a lane's two pieces of a unit of 64 k: k0 + 8 q and k0 + 32 + 8 q; a piece past K reads the row's last piece, as zeros for the weights
    auto fetch = [&](int unit, GpFrag (&x)[2], GpFrag (&wf)[NW][2]) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int k = unit * 64 + 32 * h + 8 * q;
            const int kk = min(k, K - 8);
            x[h].u = *reinterpret_cast<const gp_u32x4*>(arow + kk);
#pragma unroll
            for (int u = 0; u < NW; ++u) {
                const gp_u32x4 v = *reinterpret_cast<const gp_u32x4*>(w[u] + kk);
                wf[u][h].u = k < K ? v : zero;
            }
        }
    };
    gp_floatx4 acc[NW];
#pragma unroll
    for (int u = 0; u < NW; ++u) acc[u] = gp_floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    const int units = (K + 63) / 64;
    GpFrag xc[2], wc[NW][2];
    int unit = wave;
    if (unit < units) fetch(unit, xc, wc);
    while (unit < units) {  // (the same trips for every lane of a wave)
        const int next = unit + 4;
        GpFrag xn[2], wn[NW][2];
        if (next < units) fetch(next, xn, wn);
#pragma unroll
        for (int u = 0; u < NW; ++u) {
            acc[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wc[u][0].v, xc[0].v, acc[u], 0, 0, 0);
            acc[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wc[u][1].v, xc[1].v, acc[u], 0, 0, 0);
        }
        if (next < units) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                xc[h] = xn[h];
#pragma unroll
                for (int u = 0; u < NW; ++u) wc[u][h] = wn[u][h];
            }
        }
        unit = next;
    }
    // acc[u][r] = this wave's share of C^T[n = 4 q + r][m = i]; kept [wave][matrix][m][n]
#pragma unroll
    for (int u = 0; u < NW; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[(wave * NW + u) * 256 + i * 16 + 4 * q + r] = acc[u][r];
    __syncthreads();
    const int m = tid / 16, n = n0 + tid % 16;
    float v[2] = {0.0f, 0.0f};
#pragma unroll
    for (int u = 0; u < NW; ++u)
#pragma unroll
        for (int wv = 0; wv < 4; ++wv) v[u] += red[(wv * NW + u) * 256 + tid];
    const int id = row_id(m);
    if (id >= 0 && n < N) grouped_store<NW>(p, id, g, n, v[0], v[1]);
}

// Plain 32-bit multiply-adds: a tile of 64 rows x 64 output features, a thread 4 x 4 of them, K in
// steps of 16 through LDS. Takes every size and both element types.
template <typename T, int NW>
__global__ void __launch_bounds__(256)
grouped_plain_kernel(GroupedParams p) {
    constexpr int BK = 16;
    __shared__ float la[BK][64 + 1];
    __shared__ float lw[NW][BK][64 + 1];
    __shared__ int idx[kGroupedRows];
    const int g = grouped_rows(p, idx);
    if (g < 0) return;
    const int tid = threadIdx.x;
    const int n0 = blockIdx.y * 64;
    const int N = p.N, K = p.K;
    const T* a = static_cast<const T*>(p.a) + static_cast<int64_t>(g) * p.a_group_cols;
    const T* w[2] = {static_cast<const T*>(p.w0) + static_cast<int64_t>(g) * N * K,
                     NW == 2 ? static_cast<const T*>(p.w1) + static_cast<int64_t>(g) * N * K : nullptr};
    const int tr = (tid / 16) * 4, tc = (tid % 16) * 4;  // this thread's rows and columns of the tile
    float acc[NW][4][4];
#pragma unroll
    for (int u = 0; u < NW; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[u][i][j] = 0.0f;
    for (int k0 = 0; k0 < K; k0 += BK) {
        __syncthreads();
        // 64 x 16 values of each operand: a thread four of them, k fastest
        for (int e = tid; e < 64 * BK; e += 256) {
            const int row = e / BK, k = k0 + e % BK;
            const int id = idx[row];
            la[e % BK][row] = (id >= 0 && k < K) ? to_float<T>(a[static_cast<int64_t>(id / p.a_div) * p.lda + k]) : 0.0f;
            const int n = n0 + row;
#pragma unroll
            for (int u = 0; u < NW; ++u) lw[u][e % BK][row] = (n < N && k < K) ? to_float<T>(w[u][static_cast<int64_t>(n) * K + k]) : 0.0f;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < BK; ++k) {
            float av[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) av[i] = la[k][tr + i];
#pragma unroll
            for (int u = 0; u < NW; ++u) {
                float wv[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) wv[j] = lw[u][k][tc + j];
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc[u][i][j] = fmaf(av[i], wv[j], acc[u][i][j]);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int id = idx[tr + i];
        if (id < 0) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int n = n0 + tc + j;
            if (n < N) grouped_store<NW>(p, id, g, n, acc[0][i][j], NW == 2 ? acc[NW - 1][i][j] : 0.0f);
        }
    }
}

// The same product, bit for bit, for whole units of K (a multiple of 64): what bounds it is its chain of trips to memory, the lists, then the
// weights of the expert that they name, unit after unit. The tile's group, its rows and what the epilogue reads are asked for together, and a wave's
// units come into a ring in LDS of its own (8 rows of 64 k a load, whole cache lines), R of them in flight, waited for one by one without a barrier.
// us, cold weights, before / now: of 8 experts, 768 -> 2 x 1,536, 2 entries 6.7 / 6.3, 16 entries 11.7 / 9.5, 120 entries 16.7 / 13.4; 1,536 -> 768 16 entries
// 8.5 / 7.4, 120 12.3 / 8.7; of 16 experts, 1,600 -> 2 x 3,200, 16 entries 62 / 45; 4 rows of 12 heads, 64 -> 128 3.5 / 3.35, 128 -> 64 with a gate 3.7 / 3.55;
// 128 rows, 256 -> 512 10.4 / 7.3.
// LISTED: rows by a router's lists; FACTORS: a row's scale or a gate on the output.
template <int NW, int R, bool LISTED, bool FACTORS>
__global__ void __launch_bounds__(256)
grouped_stream_kernel(GroupedParams p) {
    constexpr int ROWS = 16 * (1 + NW), LOADS = ROWS / 8, SLOT = ROWS * 64;
    static_assert((R - 1) * LOADS <= 63, "the counter of loads in flight has six bits");
    constexpr size_t RING = static_cast<size_t>(4) * R * SLOT * 2, SUMS = 4 * NW * 256 * 4;
    __shared__ __attribute__((aligned(1024))) unsigned char lds[RING > SUMS ? RING : SUMS];
    float* const red = reinterpret_cast<float*>(lds);
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int i = lane % 16, q = lane / 16, lrow = lane / 8, lpos = lane % 8;
    const int tile = blockIdx.x, N = p.N, K = p.K, n0 = blockIdx.y * 16;
    bf16_t* const ring = reinterpret_cast<bf16_t*>(lds) + wave * R * SLOT;
    // the rows this lane brings in (places lrow and lrow + 8) and the one it stores (place tid / 16), together with the tile's group
    int g, id[2], e_id;
    if constexpr (LISTED) {
        const int* const places = p.rows_list + tile * kSkinnyRows;
        const int group = p.tile_group[tile];
        id[0] = places[lrow];
        id[1] = places[lrow + 8];
        e_id = places[tid / 16];
        g = __builtin_amdgcn_readfirstlane(group);
        if (g < 0) return;
    } else {
        const int m0 = tile * kSkinnyRows;
        g = blockIdx.z;
        id[0] = m0 + lrow < p.M ? m0 + lrow : -1;
        id[1] = m0 + lrow + 8 < p.M ? m0 + lrow + 8 : -1;
        e_id = m0 + tid / 16 < p.M ? m0 + tid / 16 : -1;
    }
    // an empty place reads the first row, a feature past N the last one: computed, never stored
    const bf16_t* from[LOADS];
#pragma unroll
    for (int l = 0; l < 2; ++l) {
        const int piece = (lpos ^ ring_swizzle(8 * l + lrow)) * 8;
        const int row = LISTED ? (id[l] >= 0 ? id[l] / p.a_div : 0) : max(id[l], 0);
        from[l] = static_cast<const bf16_t*>(p.a) + static_cast<int64_t>(row) * p.lda + static_cast<int64_t>(g) * p.a_group_cols + piece;
        const int64_t wrow = (static_cast<int64_t>(g) * N + min(n0 + 8 * l + lrow, N - 1)) * K + piece;
        from[2 + l] = static_cast<const bf16_t*>(p.w0) + wrow;
        if constexpr (NW == 2) from[4 + l] = static_cast<const bf16_t*>(p.w1) + wrow;
    }
    const int units = K / 64, mine = (units - wave + 3) / 4;  // this wave's units: wave, wave + 4, ...
    auto load = [&](int j, int slot) {  // (one past the last: the last of K again, not multiplied)
        const int k = min(wave + 4 * j, units - 1) * 64;
#pragma unroll
        for (int l = 0; l < LOADS; ++l) {
            const bf16_t* const piece = from[l] + k;
            bf16_t* const to = ring + slot * SLOT + l * 8 * 64;
            __builtin_amdgcn_global_load_lds(piece, (lds_void_ptr)to, 16, 0, 0);
        }
    };
    // what the epilogue reads, ahead of the weights; no load under a branch: who has nothing to read gets a word of the weights
    const int n = n0 + tid % 16;
    float e_scale = 1.0f, e_gate = 0.0f;
    uint32_t e_gate_word = 0;
    if constexpr (FACTORS) {
        const int row = max(e_id, 0);
        const int64_t ga = static_cast<int64_t>(row) * p.gate_stride + static_cast<int64_t>(g) * N + min(n, N - 1);
        const float* const scale_at = p.row_scale != nullptr ? p.row_scale + row : static_cast<const float*>(p.w0);
        const bf16_t* const gate16_at = p.gate != nullptr && p.gate_dtype == kBF16 ? static_cast<const bf16_t*>(p.gate) + ga : static_cast<const bf16_t*>(p.w0);
        const float* const gate32_at = p.gate != nullptr && p.gate_dtype == kF32 ? static_cast<const float*>(p.gate) + ga : static_cast<const float*>(p.w0);
        e_scale = *scale_at;
        e_gate_word = *gate16_at;
        e_gate = *gate32_at;
    }
    // (no load may cross to the other side: the waits below count on what is asked for behind them)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < R; ++t) load(t, t);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");

    gp_floatx4 acc[NW];
#pragma unroll
    for (int u = 0; u < NW; ++u) acc[u] = gp_floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    auto multiply = [&](int slot) {
        const bf16_t* const at = ring + slot * SLOT + i * 64;
        GpFrag x[2], w[NW][2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int piece = ((4 * h + q) ^ ring_swizzle(i)) * 8;
            x[h].u = *reinterpret_cast<const gp_u32x4*>(at + piece);
#pragma unroll
            for (int u = 0; u < NW; ++u) w[u][h].u = *reinterpret_cast<const gp_u32x4*>(at + 16 * (1 + u) * 64 + piece);
        }
#pragma unroll
        for (int u = 0; u < NW; ++u) {
            acc[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[u][0].v, x[0].v, acc[u], 0, 0, 0);
            acc[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[u][1].v, x[1].v, acc[u], 0, 0, 0);
        }
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
    lds_barrier();  // (the sums take the rings' place)
#pragma unroll
    for (int u = 0; u < NW; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[(wave * NW + u) * 256 + i * 16 + 4 * q + r] = acc[u][r];
    lds_barrier();
    float v[2] = {0.0f, 0.0f};
#pragma unroll
    for (int u = 0; u < NW; ++u)
#pragma unroll
        for (int wv = 0; wv < 4; ++wv) v[u] += red[(wv * NW + u) * 256 + tid];
    if (e_id < 0 || n >= N) return;
    float value = grouped_act<NW>(p, v[0], v[1]);
    if constexpr (FACTORS) {
        if (p.row_scale != nullptr) value *= e_scale;
        if (p.gate != nullptr) value *= gp_sigmoid(p.gate_dtype == kF32 ? e_gate : bf16_to_float(static_cast<bf16_t>(e_gate_word)));
    }
    const int64_t at = grouped_place(p, e_id, g) + n;
    if (p.out_dtype == kF32) static_cast<float*>(p.out)[at] = value;
    else static_cast<bf16_t*>(p.out)[at] = float_to_bf16(value);
}

template <int NW>
int launch_grouped_stream(const GroupedParams& p, const dim3& grid, hipStream_t stream) {
    const int mine = (p.K / 64 + 3) / 4;  // units a wave
    const bool factors = p.row_scale != nullptr || p.gate != nullptr;
#define LIYAB_STREAM(R)                                                                                                        \
    do {                                                                                                                       \
        if (p.rows_list != nullptr && factors) grouped_stream_kernel<NW, R, true, true><<<grid, 256, 0, stream>>>(p);          \
        else if (p.rows_list != nullptr) grouped_stream_kernel<NW, R, true, false><<<grid, 256, 0, stream>>>(p);               \
        else if (factors) grouped_stream_kernel<NW, R, false, true><<<grid, 256, 0, stream>>>(p);                              \
        else grouped_stream_kernel<NW, R, false, false><<<grid, 256, 0, stream>>>(p);                                          \
    } while (0)
    // Three units in flight, two where a unit has both halves' weights: 48 KiB of LDS, so that three workgroups share a compute unit (six units, 96 KiB and one
    // workgroup: 16 entries of 16 experts, 3,200 -> 1,600, 33 us, three 24, two 25; 2 entries of 8, 1,536 -> 768 5.4, 5.4, 5.9. Both halves, three and two: 1,600 ->
    // 2 x 3,200 49 and 45, 768 -> 2 x 768 7.0 and 7.2).
    if (mine <= 1) {
        LIYAB_STREAM(1);
    } else if constexpr (NW == 2) {
        LIYAB_STREAM(2);
    } else {
        if (mine <= 2) LIYAB_STREAM(2);
        else LIYAB_STREAM(3);
    }
#undef LIYAB_STREAM
    return check_launch("grouped_product");
}

}  // namespace liyab

using namespace liyab;

// See the head of this file. dtype: the element type of a, w0 and w1. n_groups: heads (rows_list
// null) or experts (the values of tile_group lie below it; the caller has made them so). n_tiles:
// the tiles of rows to launch (with rows_list: the length of tile_group; without: (M + block - 1) / block).
// block: the row places a tile, 64, or 16 for steps of few rows a group (bfloat16 operands in 16-byte pieces).
extern "C" int liyab_grouped_product(const void* a, int64_t lda, int a_div, int a_group_cols, const void* w0, const void* w1, int dtype,
                                     void* out, int out_dtype, int64_t ldo, int out_group_cols, const int* rows_list,
                                     const int* tile_group, int n_tiles, int block, int n_groups, const float* row_scale,
                                     const void* gate, int gate_dtype, int64_t gate_stride, int M, int N, int K, int act, int out_div, int out_extra,
                                     float limit, float slope, float shift, hipStream_t stream) {
    LIYAB_REQUIRE(a && w0 && out, "grouped_product: null pointer");
    LIYAB_REQUIRE(dtype == kF32 || dtype == kBF16, "grouped_product: unknown dtype %d", dtype);
    LIYAB_REQUIRE(out_dtype == kF32 || out_dtype == kBF16, "grouped_product: unknown output dtype %d", out_dtype);
    LIYAB_REQUIRE(M >= 0 && N > 0 && K > 0 && a_div >= 1 && n_groups >= 1 && n_groups <= 65535 && n_tiles >= 0, "grouped_product: bad sizes M=%d N=%d K=%d", M, N, K);
    LIYAB_REQUIRE((rows_list == nullptr) == (tile_group == nullptr), "grouped_product: a list of rows goes with the groups of its tiles");
    LIYAB_REQUIRE(block == kGroupedRows || block == kSkinnyRows, "grouped_product: tiles of %d rows (%d or %d)", block, kGroupedRows, kSkinnyRows);
    LIYAB_REQUIRE(rows_list != nullptr || n_tiles == (M + block - 1) / block, "grouped_product: %d tiles for %d rows", n_tiles, M);
    LIYAB_REQUIRE(gate == nullptr || gate_dtype == kF32 || gate_dtype == kBF16, "grouped_product: unknown gate dtype %d", gate_dtype);
    LIYAB_REQUIRE(gate == nullptr || gate_stride >= static_cast<int64_t>(rows_list ? 1 : n_groups) * N, "grouped_product: the gate's rows are shorter than the output's");
    LIYAB_REQUIRE((act == 0 || (act == 1 && w1 == nullptr) || (act == 2 && w1 != nullptr && limit > 0.0f)) && out_div >= 1 && out_extra >= 0, "grouped_product: activation %d is not known or does not go with these matrices", act);
    if (M == 0 || n_tiles == 0) return 0;
    GroupedParams p{a, lda, a_div, a_group_cols, w0, w1, out, ldo, out_group_cols, out_dtype, rows_list, tile_group, row_scale, gate, gate_stride, gate_dtype, M, N, K, block, act, out_div, out_extra, limit, slope, shift};
    const dim3 grid(n_tiles, (N + 63) / 64, rows_list ? 1 : n_groups);
    const bool matrix = dtype == kBF16 && K % 8 == 0 && lda % 8 == 0 && a_group_cols % 8 == 0 &&
                        (reinterpret_cast<uintptr_t>(a) & 15) == 0 && (reinterpret_cast<uintptr_t>(w0) & 15) == 0 &&
                        (reinterpret_cast<uintptr_t>(w1) & 15) == 0;
    LIYAB_REQUIRE(block == kGroupedRows || matrix, "grouped_product: tiles of %d rows are for bfloat16 operands in 16-byte pieces", kSkinnyRows);
    if (block == kSkinnyRows) {
        const dim3 skinny(n_tiles, (N + 15) / 16, rows_list ? 1 : n_groups);
        // (lists with a single unit of K have nothing to stream: the kernel of registers, 8 experts, 60 tokens, 64 -> 2 x 64 3.3 us against 3.55; a step's heads are as fast or
        // faster by rings, 64 -> 128 3.35 against 3.5)
        if (K % 64 == 0 && (K > 64 || rows_list == nullptr)) return w1 != nullptr ? launch_grouped_stream<2>(p, skinny, stream) : launch_grouped_stream<1>(p, skinny, stream);
        if (w1 != nullptr) grouped_skinny_kernel<2><<<skinny, 256, 0, stream>>>(p);
        else grouped_skinny_kernel<1><<<skinny, 256, 0, stream>>>(p);
    } else if (matrix && K % 64 == 0 && (w1 == nullptr || gate == nullptr) && static_cast<int64_t>(n_tiles) * grid.y * grid.z < (1 << 24)) {
        // (its tiles lie along one dimension of the grid, which holds less than 2^32 threads: larger grids, of mostly spare tiles, go to the kernel below)
        // Short inner sizes are prologue and epilogue: narrow tiles and more workgroups a compute unit (heads of 128 -> 64 with a gate, 4,000 rows: 18.1 us in
        // tiles of 128 features, half of them outside, 9.1 in 64); long ones a wide tile (3,280 entries, 1,536 -> 768: 22.7 us in three stages, 25.7 in
        // two). Two matrices: two stages, three workgroups a unit (768 -> 2 x 1,536: 35.3 us, 41.5 in three; 600 entries 15.3 and 14.9).
        const int groups = rows_list ? 1 : n_groups;
        if (w1 != nullptr) return launch_grouped_tile<2, 128, 2>(p, n_tiles, groups, stream);
        return K >= 768 && N > 64 ? launch_grouped_tile<1, 128, 3>(p, n_tiles, groups, stream) : launch_grouped_tile<1, 64, 2>(p, n_tiles, groups, stream);
    } else if (matrix) {
        if (w1 != nullptr) grouped_mfma_kernel<2><<<grid, 256, 0, stream>>>(p);
        else grouped_mfma_kernel<1><<<grid, 256, 0, stream>>>(p);
    } else if (dtype == kBF16) {
        if (w1 != nullptr) grouped_plain_kernel<bf16_t, 2><<<grid, 256, 0, stream>>>(p);
        else grouped_plain_kernel<bf16_t, 1><<<grid, 256, 0, stream>>>(p);
    } else {
        if (w1 != nullptr) grouped_plain_kernel<float, 2><<<grid, 256, 0, stream>>>(p);
        else grouped_plain_kernel<float, 1><<<grid, 256, 0, stream>>>(p);
    }
    return check_launch("grouped_product");
}
