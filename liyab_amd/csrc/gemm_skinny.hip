// out[M,N] = a[M,K] . w[N,K]^T in bfloat16 for steps of few tokens (M <= 64):
// decoding, where the product is a stream of the weights.
//
// A workgroup owns 16 * NT output features (rows of `w`) and all M tokens as
// MT tiles of 16; its waves split K and add their partial sums through LDS in
// wave order. With v_mfma_f32_16x16x32_bf16 the weights are the first
// operand (16 rows) and the tokens the second (16), so an accumulator is a
// transposed output tile. A lane holds 8 consecutive k of its row per
// instruction, the four lane groups of a row 32 consecutive k: one load
// instruction reads 64 contiguous bytes of each of 16 rows (whole sectors;
// a lane reading 32 contiguous bytes in two instructions touched every
// sector twice). Weights are
// read, where K is whole units of 64 by way of a ring in LDS of each wave's own
// (gemm_stream_kernel), otherwise straight from global memory into registers, 16 bytes a lane,
// one trip ahead of the multiplies; the tokens' rows come from L2 (every
// workgroup reads all of them: few, wide tiles of N would starve most CUs).
// K must be a multiple of 8. The order of the sum depends on the output feature, K and the
// split only, never on M.
//
// The product may be cut over K into parts (blockIdx.z), each part's sums going to its own
// plane of 32-bit sums; the first plane may take the bias and the rows the product is to be
// added to (themselves a sum of planes), so that the planes together are the new rows.
#include "common.h"
#include "launchers.h"
#include "epilogue.h"
#include "ring.h"

namespace liyab {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float floatx4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

union Frag {
    u32x4 u;
    bf16x8 v;
};

// What the first part of a product cut over K adds to its plane: the rows the product is
// added to, given as a sum of planes [n][M][N] (added in their order), or nothing.
struct BaseSum {
    const float* planes;
    int n;
    int64_t stride;
};

template <typename OutT, int MT, int NT, int MAXW>
__global__ void __launch_bounds__(64 * MAXW)
gemm_skinny_kernel(const bf16_t* __restrict__ a, int64_t lda, const bf16_t* __restrict__ w, int M, int N, int K,
                   EpiParams epi, BaseSum base, int part_k, int64_t part_stride) {
    constexpr int UPT = (MT * NT == 1) ? 2 : 1;  // units of 64 k per trip
    constexpr int TILES = MT * NT;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int ksplit = blockDim.x / 64;
    float* red = reinterpret_cast<float*>(smem);

    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    const int i = lane % 16, g = lane / 16;
    const int n0 = blockIdx.x * 16 * NT;
    const int m0 = blockIdx.y * 16 * MT;  // this workgroup's rows: [m0, m0 + 16 MT) of M
    // K may be cut into parts of part_k (a multiple of 64) over blockIdx.z, each part's sums
    // going to its own plane of the output; this workgroup's k are [k_begin, k_end)
    const int k_begin = blockIdx.z * part_k, k_end = min(K, k_begin + part_k);
    const int units = (k_end - k_begin + 63) / 64;
    if (gridDim.z > 1) epi.out = static_cast<float*>(epi.out) + blockIdx.z * part_stride;
    if (blockIdx.z > 0) epi.bias = nullptr;  // a cut product's bias goes to its first plane only
    const u32x4 zero = {0, 0, 0, 0};
    const bf16_t* wrow[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) wrow[t] = w + static_cast<int64_t>(min(n0 + 16 * t + i, N - 1)) * K;

    // 8 consecutive k of a row; past the end it is the last piece, read and dropped: a load under
    // a branch would make the compiler wait for every load in flight, the next trip's too
    auto piece = [&](const bf16_t* row, int k) {
        const u32x4 v = *reinterpret_cast<const u32x4*>(row + min(k, k_end - 8));
        return k < k_end ? v : zero;
    };
    // unit u covers k in k_begin + [64 u, 64 u + 64): two instructions of 32 k, this lane's 8 start at 8 g
    auto load_w = [&](int u0, Frag (&f)[UPT][NT][2]) {
#pragma unroll
        for (int p = 0; p < UPT; ++p) {
            const int k = k_begin + (u0 + p) * 64 + g * 8;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                f[p][t][0].u = piece(wrow[t], k);
                f[p][t][1].u = piece(wrow[t], k + 32);
            }
        }
    };
    // How K goes to the waves. As a rule a trip of the workgroup is UPT * ksplit consecutive
    // units, one wave after the other, and the next trip the next such stretch. Where rows lie
    // a multiple of 32 KB apart (K a multiple of 16,384), the sixteen rows of a workgroup, and
    // every workgroup's, begin in the same few memory channels, and workgroups in step crowd
    // those: there a wave walks a block of consecutive trips of its own, and a workgroup starts
    // blockIdx.x mod trips trips into its blocks and goes round past their end (16,384 ->
    // 4,096 in a decode step: 34.3 -> 28.3 us; at rows of 8 KB the same walk is no faster in
    // a step, though up to 12 % faster alone). The order of a sum depends on the output
    // feature, K and the split only, never on M.
    const bool blocks = K % 16384 == 0;
    const int trips = max(1, (units + UPT * ksplit - 1) / (UPT * ksplit));
    int trip = blocks ? static_cast<int>(blockIdx.x % trips) : 0;
    auto unit_of = [&](int t) { return blocks ? (wave * trips + t) * UPT : (t * ksplit + wave) * UPT; };
    Frag wc[UPT][NT][2];
    load_w(unit_of(trip), wc);
    // what the epilogue will read for this thread's first output (bias, residual) is asked for
    // now: after the sums it would be one more trip to memory on the critical path
    const int e_m = m0 + 16 * ((tid / 256) / NT) + (tid % 256) / 16, e_n = n0 + 16 * ((tid / 256) % NT) + tid % 16;
    const bool e_mine = tid < TILES * 256 && e_m < M && e_n < N;
    const float e_bias = (e_mine && epi.bias != nullptr) ? epi.bias[e_n] : 0.0f;
    const float e_res = (e_mine && epi.mode == kEpiResidual) ? epi.residual[static_cast<int64_t>(e_m) * epi.ldr + e_n] : 0.0f;
    // the first part's share of the rows the product is added to: up to four planes asked for
    // together (a plane past the last is the last one again, read and dropped)
    const bool based = base.planes != nullptr && blockIdx.z == 0;
    float e_base[4];
    {
        // no branch around the loads (a load under a branch is waited for where the branch ends,
        // and the weights asked for above with it): whoever has nothing to add reads a word of
        // the weights instead and drops it
        const float* src = based ? base.planes : reinterpret_cast<const float*>(w);
        const int64_t at = (based && e_mine) ? static_cast<int64_t>(e_m) * N + e_n : 0;
        const int64_t stride = based ? base.stride : 0;
        const int last = based ? base.n - 1 : 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) e_base[q] = src[min(q, last) * stride + at];
    }
    __builtin_amdgcn_sched_barrier(0);  // keep the loads here: the scheduler would sink them to their use

    const bf16_t* arow[MT];
#pragma unroll
    for (int s = 0; s < MT; ++s) arow[s] = a + static_cast<int64_t>(min(m0 + 16 * s + i, M - 1)) * lda;
    // the tokens' fragments travel with the weights', a trip ahead: asked for after the next
    // trip's weights they would make every trip wait for those too (loads return in order)
    auto load_x = [&](int u0, Frag (&x)[UPT][MT][2]) {
#pragma unroll
        for (int p = 0; p < UPT; ++p) {
            const int k = k_begin + (u0 + p) * 64 + g * 8;
#pragma unroll
            for (int s = 0; s < MT; ++s) {
                x[p][s][0].u = piece(arow[s], k);
                x[p][s][1].u = piece(arow[s], k + 32);
            }
        }
    };
    Frag xc[UPT][MT][2];
    load_x(unit_of(trip), xc);

    floatx4 acc[MT][NT];
#pragma unroll
    for (int s = 0; s < MT; ++s)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[s][t] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};

    auto multiply = [&]() {
#pragma unroll
        for (int p = 0; p < UPT; ++p)
#pragma unroll
            for (int s = 0; s < MT; ++s)
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    acc[s][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wc[p][t][0].v, xc[p][s][0].v, acc[s][t], 0, 0, 0);
                    acc[s][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wc[p][t][1].v, xc[p][s][1].v, acc[s][t], 0, 0, 0);
                }
    };
    // every trip but the last asks for the next trip's operands before it multiplies; the last
    // one is peeled off, so no trip asks for (and then waits for) operands nobody uses
    // (dealt trip by trip, a wave whose unit of the last trip lies past the end of K stops a trip
    // early: it would ask for the rows' last bytes again, as every such wave would, and drop them)
    const int my_trips = blocks ? trips : max(1, (units - wave * UPT + UPT * ksplit - 1) / (UPT * ksplit));
    for (int left = my_trips - 1; left > 0; --left) {
        trip = trip + 1 == trips ? 0 : trip + 1;
        Frag wn[UPT][NT][2], xn[UPT][MT][2];
        load_w(unit_of(trip), wn);
        load_x(unit_of(trip), xn);
        multiply();
#pragma unroll
        for (int p = 0; p < UPT; ++p) {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                wc[p][t][0] = wn[p][t][0];
                wc[p][t][1] = wn[p][t][1];
            }
#pragma unroll
            for (int s = 0; s < MT; ++s) {
                xc[p][s][0] = xn[p][s][0];
                xc[p][s][1] = xn[p][s][1];
            }
        }
    }
    multiply();  // a wave past the end of K holds zeros
    // acc[s][t][r] = partial C^T[n = 16 t + 4 g + r][m = 16 s + i]; kept [tile][m][n] per wave
#pragma unroll
    for (int s = 0; s < MT; ++s)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[(wave * TILES + s * NT + t) * 256 + i * 16 + 4 * g + r] = acc[s][t][r];
    __syncthreads();
    for (int e = tid; e < TILES * 256; e += blockDim.x) {
        const int tile = e / 256, s = tile / NT, t = tile % NT;
        const int m = m0 + 16 * s + (e % 256) / 16, n = n0 + 16 * t + e % 16;
        float v = 0.0f;
        for (int q = 0; q < ksplit; ++q) v += red[q * TILES * 256 + e];
        if (m >= M || n >= N) continue;
        if (based) {
            // this plane = (sums + bias) + (base planes added up in their order)
            const float* bp = base.planes + static_cast<int64_t>(m) * N + n;
            float b;
            if (e == tid) {
                b = e_base[0];
#pragma unroll
                for (int q = 1; q < 4; ++q)
                    if (q < base.n) b += e_base[q];
                for (int q = 4; q < base.n; ++q) b += bp[q * base.stride];
            } else {
                b = bp[0];
                for (int q = 1; q < base.n; ++q) b += bp[q * base.stride];
            }
            v = (v + (e == tid ? e_bias : epilogue_bias(epi, n))) + b;
            static_cast<float*>(epi.out)[static_cast<int64_t>(m) * epi.ldo + n] = v;
            continue;
        }
        if (e != tid) epilogue_store<OutT>(epi, m, n, v);
        else if (epi.mode == kEpiResidual) epi.residual[static_cast<int64_t>(m) * epi.ldr + n] = e_res + (v + e_bias);
        else epilogue_store_biased<OutT>(epi, m, n, v + e_bias);
    }
}

// The same product, bit for bit, for one tile of 16 rows a workgroup, 16 or 32 features and whole units of K (a multiple of 64, and not of 16,384): a
// wave's units reach it through a ring in LDS of its own, 8 rows of 64 k a load (global_load_lds, whole cache lines), with no barrier: a wave waits
// for its own loads. What bounds a product of this size is a chain: the first trip to memory, and what stands behind it. Straight into registers a
// load touched 16 rows' sectors and an operand of 8 rows was read for 16; the waves' sums were read one by one; and waves without a unit of K
// were launched. The waves, each wave's units and the order of the sums are those of gemm_skinny_kernel. The epilogue is fixed at compile time: a
// kernel this short waits for its own instructions, cold in every launch of a chain (all epilogues in one, 1,300 instructions and not 500: 768 -> 768
// 3.8 us and not 3.3). us, cold weights, before / now: 8 rows 768 -> 768 4.5 / 3.3, -> 3,072 5.2 / 4.1, -> 50,257 22.1 / 16.7, 3,072 -> 768 8.0 / 4.9, in
// four parts 5.3 / 4.3, 1,600 -> 6,400 8.9 / 6.3; 16 rows 768 -> 768 4.8 / 3.4, 1,600 -> 4,800 9.7 / 5.8.
// MR: rows of the ring, 8 or 16, M rounded up (the matrix operand's other rows repeat the last). NT: tiles of 16 features. R: units of the ring.
constexpr int kUnit = 64;

// EPI: an epilogue fixed at compile time: none, residual, kEpiPlanes (planes with rows to add to), or a gated feed-forward's first product, kEpiGlu* (w = the
// gate's N rows, then the other half's: a workgroup takes 16 features of both, and their 32-bit sums meet in act(gate) * other, as in
// elementwise_norms.hip's kernel, whose link in the chain and trip through memory go); -1 reads it from the parameters.
constexpr int kEpiPlanes = 5, kEpiGluSilu = 6, kEpiGluGelu = 7;
template <typename OutT, int MR, int NT, int R, int EPI>
__global__ void __launch_bounds__(1024, R == 1 ? 8 : 4)  // one unit in flight: two workgroups of 16 waves a compute unit
gemm_stream_kernel(const bf16_t* __restrict__ a, int64_t lda, const bf16_t* __restrict__ w, int M, int N, int K,
                   EpiParams epi, BaseSum base, int part_k, int64_t part_stride, int split_shift, int trip_shift) {
    constexpr bool GLU = EPI == kEpiGluSilu || EPI == kEpiGluGelu;
    static_assert(!GLU || NT == 2, "one tile of the gate's features and one of the other half's");
    constexpr int NB = 16 * NT, LOADS = (NB + MR) / 8, SLOT = (NB + MR) * kUnit;
    static_assert((R - 1) * LOADS <= 63, "the counter of loads in flight has six bits");
    extern __shared__ __attribute__((aligned(1024))) unsigned char stream_lds[];
    float* const red = reinterpret_cast<float*>(stream_lds);  // [wave][NT][256], once the rings have been read
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64), waves = blockDim.x / 64;
    const int i = lane % 16, g = lane / 16;
    const int n0 = blockIdx.x * (GLU ? 16 : NB), m0 = blockIdx.y * 16;
    const int k_begin = blockIdx.z * part_k, k_end = min(K, k_begin + part_k);
    // this wave's units: those of trips wave, wave + ksplit, ..., of one or two units each (the last of all may be half a pair); ksplit = 1 << split_shift
    const int per_trip = 1 << trip_shift, ksplit = 1 << split_shift;
    const int units = (k_end - k_begin) / kUnit, trips = (units + per_trip - 1) >> trip_shift;
    const int my_trips = wave < ksplit ? (trips - wave + ksplit - 1) >> split_shift : 0;
    const int mine = (my_trips << trip_shift) - ((units & (per_trip - 1)) != 0 && ((trips - 1) & (ksplit - 1)) == wave ? 1 : 0);
    if (gridDim.z > 1) epi.out = static_cast<float*>(epi.out) + blockIdx.z * part_stride;
    if (blockIdx.z > 0) epi.bias = nullptr;  // a cut product's bias goes to its first plane only
    bf16_t* const ring = reinterpret_cast<bf16_t*>(stream_lds) + wave * R * SLOT;

    const int lrow = lane / 8, lpos = lane % 8;  // this lane's part in a load
    const bf16_t* from[LOADS];
#pragma unroll
    for (int l = 0; l < 2 * NT; ++l) {
        const int row = GLU && l >= 2 ? N + min(n0 + 8 * (l - 2) + lrow, N - 1) : min(n0 + 8 * l + lrow, N - 1);
        from[l] = w + static_cast<int64_t>(row) * K + k_begin + (lpos ^ ring_swizzle(8 * l + lrow)) * 8;
    }
#pragma unroll
    for (int l = 2 * NT; l < LOADS; ++l) {
        const int row = 8 * (l - 2 * NT) + lrow;
        from[l] = a + static_cast<int64_t>(min(m0 + row, M - 1)) * lda + k_begin + (lpos ^ ring_swizzle(row)) * 8;
    }
    auto load = [&](int j, int slot) {  // unit j of this wave's (one past its last: the last of K, not multiplied)
        const int k = min(((((j >> trip_shift) << split_shift) + wave) << trip_shift) + (j & (per_trip - 1)), units - 1) * kUnit;
#pragma unroll
        for (int l = 0; l < LOADS; ++l) {
            const bf16_t* const piece = from[l] + k;
            bf16_t* const to = ring + slot * SLOT + l * 8 * kUnit;
            __builtin_amdgcn_global_load_lds(piece, (lds_void_ptr)to, 16, 0, 0);
        }
    };
    // What the epilogue reads for this thread's first output is asked for first of all (counted in order, and the weights are waited for unit by
    // unit), with no load under a branch: who has nothing to read gets a word of the weights. The first part's share of the rows the product is
    // added to: up to four planes (a plane past the last is the last one again, dropped).
    typedef const __attribute__((address_space(1))) float* global_floats;
    const int e_m = min(m0 + (tid % 256) / 16, M - 1), e_n = min(n0 + 16 * (tid / 256 % NT) + tid % 16, N - 1);
    const bool based = EPI == kEpiPlanes && blockIdx.z == 0;
    const auto nothing = (global_floats)(w);
    auto bias_at = epi.bias != nullptr ? (global_floats)(epi.bias + e_n) : nothing;
    auto res_at = based                        ? (global_floats)(base.planes + static_cast<int64_t>(e_m) * N + e_n)
                  : (EPI < 0 ? epi.mode : EPI) == kEpiResidual ? (global_floats)(epi.residual + static_cast<int64_t>(e_m) * epi.ldr + e_n)
                                             : nothing;
    const int64_t base_stride = based ? base.stride : 0;
    const int base_last = based ? base.n - 1 : 0;
    asm volatile("" : "+v"(bias_at), "+v"(res_at));  // (worked out here, ahead of every load)
    const float e_bias = GLU ? 0.0f : *bias_at;
    float e_res[4];
#pragma unroll
    for (int q = 0; q < (EPI == kEpiPlanes ? 4 : 1); ++q) e_res[q] = EPI == kEpiNone || GLU ? 0.0f : res_at[min(q, base_last) * base_stride];
    // (no load may cross to the other side: the waits below count on what is asked for behind them)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int p = 0; p < R; ++p) load(p, p);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");

    floatx4 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    const int arow = min(i, M - 1 - m0);
    auto multiply = [&](int slot) {
        const bf16_t* const sw = ring + slot * SLOT + i * kUnit;
        const bf16_t* const sa = ring + slot * SLOT + (NB + arow) * kUnit;
        Frag x[NT][2], y[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int t = 0; t < NT; ++t) x[t][h].u = *reinterpret_cast<const u32x4*>(sw + 16 * t * kUnit + ((4 * h + g) ^ ring_swizzle(i)) * 8);
            y[h].u = *reinterpret_cast<const u32x4*>(sa + ((4 * h + g) ^ ring_swizzle(arow)) * 8);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[t][h].v, y[h].v, acc[t], 0, 0, 0);
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
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[(wave * NT + t) * 256 + i * 16 + 4 * g + r] = acc[t][r];
    lds_barrier();
    if constexpr (GLU) {
        for (int e = tid; e < 256; e += blockDim.x) {
            const int m = m0 + e / 16, n = n0 + e % 16;
            if (m >= M || n >= N) continue;
            float v[2] = {0.0f, 0.0f};
            for (int q = 0; q < waves; ++q)
#pragma unroll
                for (int t = 0; t < 2; ++t) v[t] += red[(q * 2 + t) * 256 + e];
            const float act = EPI == kEpiGluSilu ? v[0] * (1.0f / (1.0f + expf(-v[0]))) : gelu_tanh_fast(v[0]);
            static_cast<OutT*>(epi.out)[static_cast<int64_t>(m) * epi.ldo + n] = from_float<OutT>(act * v[1]);
        }
        return;
    }
    for (int e = tid; e < NT * 256; e += blockDim.x) {
        const int m = m0 + e % 256 / 16, n = n0 + 16 * (e / 256) + e % 16;
        if (m >= M || n >= N) continue;
        float v = 0.0f;
        for (int q0 = 0; q0 < waves; q0 += 8) {
            float s[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) s[q] = red[min(q0 + q, waves - 1) * NT * 256 + e];
#pragma unroll
            for (int q = 0; q < 8; ++q) v += q0 + q < waves ? s[q] : 0.0f;
        }
        const bool first = e == tid;
        const float bias = first ? (epi.bias != nullptr ? e_bias : 0.0f) : epilogue_bias(epi, n);
        if (based) {
            // this plane = (sums + bias) + (base planes added up in their order)
            const float* bp = base.planes + static_cast<int64_t>(m) * N + n;
            float b = first ? e_res[0] : bp[0];
#pragma unroll
            for (int q = 1; q < 4; ++q)
                if (q < base.n) b += first ? e_res[q] : bp[q * base.stride];
            for (int q = 4; q < base.n; ++q) b += bp[q * base.stride];
            static_cast<float*>(epi.out)[static_cast<int64_t>(m) * epi.ldo + n] = (v + bias) + b;
        } else if (first && (EPI < 0 ? epi.mode : EPI) == kEpiResidual) {
            epi.residual[static_cast<int64_t>(m) * epi.ldr + n] = e_res[0] + (v + bias);
        } else {
            epilogue_store_biased<OutT, EPI == kEpiPlanes ? kEpiNone : EPI>(epi, m, n, v + bias);
        }
    }
}

template <typename OutT, int MR, int NT, int R, int EPI>
int launch_stream_as(const bf16_t* a, int64_t lda, const bf16_t* w, int M, int N, int K, int ksplit, int waves, const EpiParams& epi, const BaseSum& base,
                     int kparts, int part_k, int64_t part_stride, int trip_shift, hipStream_t stream) {
    size_t smem = static_cast<size_t>(waves) * R * (16 * NT + MR) * kUnit * sizeof(bf16_t);
    if (smem < waves * NT * 256 * sizeof(float)) smem = waves * NT * 256 * sizeof(float);
    LIYAB_REQUIRE(smem <= 160 * 1024, "gemm_skinny: %zu bytes of LDS", smem);
    auto kern = gemm_stream_kernel<OutT, MR, NT, R, EPI>;
    static bool ready = false;  // once per instantiation, outside any stream capture's first use
    if (!ready) {
        hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        ready = true;
    }
    constexpr int wide = EPI >= kEpiGluSilu ? 16 : 16 * NT;  // output features a workgroup
    kern<<<dim3((N + wide - 1) / wide, (M + 15) / 16, kparts), 64 * waves, smem, stream>>>(a, lda, w, M, N, K, epi, base, part_k, part_stride, __builtin_ctz(ksplit), trip_shift);
    return check_launch("gemm_skinny");
}
template <typename OutT, int EPI>
int launch_stream_epi(const void* a, int64_t lda, const void* w, int M, int N, int K, int ksplit, const EpiParams& epi, const BaseSum& base, int kparts,
                  int64_t part_stride, int trip_shift, hipStream_t stream) {
    const int per_trip = 1 << trip_shift, units = (K / kUnit + kparts - 1) / kparts;
    const int trips = (units + per_trip - 1) / per_trip, mine = per_trip * ((trips + ksplit - 1) / ksplit);  // units of a part, units a wave
    const int rows = M <= 8 ? 8 : 16;
    int waves = ksplit < trips ? ksplit : trips;
    auto ring = [&](int nt, int r) { return static_cast<size_t>(waves) * r * (16 * nt + rows) * kUnit * 2; };
    const int64_t strips = static_cast<int64_t>((N + 15) / 16) * ((M + 15) / 16) * kparts;
    // With a few more strips than compute units a workgroup takes two, where their rings fit: one strip's rings of eight waves, four units in flight, leave a compute unit
    // no room for another workgroup, and the strips past 256 would wait for a second round (8 rows, us by one strip / by two: 1,280 -> 5,120 7.3 / 5.7, 1,600 -> 6,144 8.1 /
    // 6.6, 3,072 -> 7,168 12.4 / 10.4; 16 rows 6.6 / 6.0, 7.5 / 6.9, 11.7 / 10.8; up to 1,024 even). With up to twice as many it does where eight waves still share K (1,920 ->
    // 7,680 9.6 / 8.4, 2,304 -> 8,192 11.1 / 9.8, 3,072 -> 8,192 13.1 / 11.7), not with four, whose rings share a unit (8,177 features on, up to 2,240 long: 1,664 -> 8,192
    // 7.5 / 8.0, 2,048 -> 8,192 9.1 / 9.8). Beyond, the bytes are the bound (1,600 -> 10,240 9.3 / 10.5, 4,096 -> 7,168 14.4 / 14.7, -> 8,192 15.4 / 16.8)
    const bool wide = trip_shift == 1 && strips > 256 && strips <= (K > 1600 && K <= 3072 && ksplit > 4 ? 512 : 448) && ring(2, 2) <= 160 * 1024;
    const int nt = wide ? 2 : 1;
    // a thread an output element at least, so that each has what its epilogue reads asked for ahead (waves without a unit of K bring in one again)
    if (strips <= 256 && waves < 4 * nt && ring(nt, 2) * 4 * nt / waves <= 160 * 1024) waves = 4 * nt;
    // four units in flight where a wave has more than two and the rings leave a compute unit room for others
    const bool four = mine > 2 && ring(nt, 4) <= 96 * 1024;
    auto* pa = static_cast<const bf16_t*>(a);
    auto* pw = static_cast<const bf16_t*>(w);
#define LIYAB_STREAM(MR, NT, R) launch_stream_as<OutT, MR, NT, R, EPI>(pa, lda, pw, M, N, K, ksplit, waves, epi, base, kparts, units * kUnit, part_stride, trip_shift, stream)
    // more workgroups than compute units, of a wave a unit or two: one unit in flight, so that two of them share a compute unit (48 rows, us, two in flight and
    // one: 768 -> 2,304 6.5 and 5.0, -> 3,072 8.6 and 6.0, 1,600 -> 1,600 7.4 and 6.2)
    if (trip_shift == 0 && strips > 256 && mine <= 2 && ring(1, 2) > 80 * 1024) {
        // (two of 16 waves share one as long as a wave has 64 registers, which a kernel that reads its epilogue from the parameters passes by 12: each has a kernel of its own. us, 17
        // and 24 rows, 1,280 -> 3,840 with GELU, one kernel / its own 7.2 / 6.2, 7.1 / 6.2)
#define LIYAB_FIXED(E) launch_stream_as<OutT, 16, 1, 1, E>(pa, lda, pw, M, N, K, ksplit, waves, epi, base, kparts, units * kUnit, part_stride, trip_shift, stream)
        if constexpr (EPI >= 0) return LIYAB_FIXED(EPI);
        else if (epi.mode == kEpiGeluTanh) return LIYAB_FIXED(kEpiGeluTanh);
        else if (epi.mode == kEpiGeluErf) return LIYAB_FIXED(kEpiGeluErf);
        else return LIYAB_FIXED(kEpiQkvPaged);
#undef LIYAB_FIXED
    }
    if (rows == 8) {
        if (wide) return four ? LIYAB_STREAM(8, 2, 4) : LIYAB_STREAM(8, 2, 2);
        return four ? LIYAB_STREAM(8, 1, 4) : LIYAB_STREAM(8, 1, 2);
    }
    if (wide) return four ? LIYAB_STREAM(16, 2, 4) : LIYAB_STREAM(16, 2, 2);
    return four ? LIYAB_STREAM(16, 1, 4) : LIYAB_STREAM(16, 1, 2);
#undef LIYAB_STREAM
}
int launch_stream(const void* a, int64_t lda, const void* w, int M, int N, int K, int ksplit, const EpiParams& epi, const BaseSum& base, int kparts,
                  int64_t part_stride, int trip_shift, hipStream_t stream) {
#define LIYAB_STREAM(OUT, EPI) launch_stream_epi<OUT, EPI>(a, lda, w, M, N, K, ksplit, epi, base, kparts, part_stride, trip_shift, stream)
    if (base.planes != nullptr) return LIYAB_STREAM(float, kEpiPlanes);
    if (epi.mode == kEpiResidual) return LIYAB_STREAM(float, kEpiResidual);
    if (epi.out_dtype == kF32) return epi.mode == kEpiNone ? LIYAB_STREAM(float, kEpiNone) : LIYAB_STREAM(float, -1);
    return epi.mode == kEpiNone ? LIYAB_STREAM(bf16_t, kEpiNone) : LIYAB_STREAM(bf16_t, -1);
#undef LIYAB_STREAM
}
template <int MT, int NT, int MAXW>
int launch_skinny(const void* a, int64_t lda, const void* w, int M, int N, int K, int ksplit, const EpiParams& epi,
                  const BaseSum& base, int kparts, int64_t part_stride, hipStream_t stream) {
    // K in kparts parts, each a whole number of units of 64 and none of them empty (the caller's check)
    const int part_k = ((K + 63) / 64 + kparts - 1) / kparts * 64;
    const dim3 grid((N + 16 * NT - 1) / (16 * NT), (M + 16 * MT - 1) / (16 * MT), kparts);
    auto* pa = static_cast<const bf16_t*>(a);
    auto* pw = static_cast<const bf16_t*>(w);
    if (ksplit > MAXW) ksplit = MAXW;
    size_t smem = static_cast<size_t>(ksplit) * MT * NT * 256 * sizeof(float);
    const bool f32 = epi.mode == kEpiResidual || epi.out_dtype == kF32;
    if (f32) {
        auto kern = gemm_skinny_kernel<float, MT, NT, MAXW>;
        static bool ready = false;
        if (!ready) {
            hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
            ready = true;
        }
        kern<<<grid, 64 * ksplit, smem, stream>>>(pa, lda, pw, M, N, K, epi, base, part_k, part_stride);
    } else {
        auto kern = gemm_skinny_kernel<bf16_t, MT, NT, MAXW>;
        static bool ready = false;
        if (!ready) {
            hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
            ready = true;
        }
        kern<<<grid, 64 * ksplit, smem, stream>>>(pa, lda, pw, M, N, K, epi, base, part_k, part_stride);
    }
    return check_launch("gemm_skinny");
}

// Waves that share K: until each has one trip's worth of it (everything is then asked for at once),
// or they cover the chip several times over.
static int choose_ksplit(int tiles, int units, int per_trip) {
    int ksplit = 1;
    // (with so many output features that one wave a workgroup covers the chip, two or four
    // still pay while a wave keeps more than 8 units: 18.3 against 20.0 us for 768 -> 50,257)
    while (ksplit < 16 && units > ksplit * per_trip && (tiles * ksplit < 2048 || units / ksplit > 8)) ksplit *= 2;
    return ksplit;
}

static int skinny_dispatch(const void* a, int64_t lda, const void* w, int M, int N, int K, int ksplit, int wide, int mtile,
                           const EpiParams& epi, const BaseSum& base, hipStream_t stream, int kparts = 1,
                           int64_t part_stride = 0) {
    // tiles of 16 rows a workgroup: all of M in one workgroup reads the weights once; with few
    // output features that leaves most of the chip idle, and the rows are spread over workgroups
    // instead (the weights then come from L2 after their first reading)
    // (measured at 24 to 64 rows over GPT-2 small's, medium's and XL's shapes: the most rows a
    // workgroup that still leaves 144 workgroups or more is the fastest or close to it)
    int mt = 1;
    if (mtile > 0) {
        mt = mtile;
    } else {
        const int strips = (N + 15) / 16;
        for (int cand = M <= 16 ? 1 : (M <= 32 ? 2 : 4); cand > 1; cand /= 2)
            if (strips * ((M + 16 * cand - 1) / (16 * cand)) >= 144) {
                mt = cand;
                break;
            }
    }
    LIYAB_REQUIRE(mt == 1 || mt == 2 || mt == 4, "gemm_skinny: %d tiles of rows a workgroup is not 1, 2 or 4", mt);
    // wide tiles of N (64 features a workgroup) when N is so large that every workgroup
    // re-reading the tokens would cost more than the weights
    if (wide < 0) wide = (mt > 1 && static_cast<long>(N) * M > (1L << 20)) ? 1 : 0;
    const int nt = wide ? 4 : 1;
    if (ksplit == 0) {
        const int tiles = ((N + 16 * nt - 1) / (16 * nt)) * ((M + 16 * mt - 1) / (16 * mt)) * kparts;
        ksplit = choose_ksplit(tiles, ((K + 63) / 64 + kparts - 1) / kparts, mt * nt == 1 ? 2 : 1);
    }
    LIYAB_REQUIRE(ksplit == 1 || ksplit == 2 || ksplit == 4 || ksplit == 8 || ksplit == 16,
                  "gemm_skinny: ksplit %d is not 1, 2, 4, 8 or 16", ksplit);
    // (with one or two units of K and more strips than compute units the kernel of registers is as fast, 128 -> 8,192 at one row 3.8 us against 3.9)
    if (nt == 1 && mt == 1 && K % kUnit == 0 && K % 16384 != 0 && (K > 2 * kUnit || N * ((M + 15) / 16) <= 16 * 256)) {
        return launch_stream(a, lda, w, M, N, K, ksplit, epi, base, kparts, part_stride, 1, stream);
    }
    // More rows than 16: blocks of 16, each reading the weights again (from L2 but for the first), with the waves and the order of sums of the tiles of rows
    // chosen above. (us, cold weights, registers / rings: 24 rows 768 -> 768 4.9 / 3.4, -> 3,072 6.3 / 5.0, 3,072 -> 768 9.0 / 5.5, 6,400 -> 1,600 15.1 / 10.1; 64 rows
    // 768 -> 768 5.0 / 3.6, -> 2,304 8.3 / 5.9, 1,600 -> 1,600 8.0 / 6.4, -> 4,800 17.8 / 12.0, 2,048 -> 8,192 24.6 / 20.8.)
    if (nt == 1 && mt > 1 && K % kUnit == 0 && K % 16384 != 0) return launch_stream(a, lda, w, M, N, K, ksplit, epi, base, kparts, part_stride, 0, stream);
    if (nt == 1) {
        if (mt == 1) return launch_skinny<1, 1, 16>(a, lda, w, M, N, K, ksplit, epi, base, kparts, part_stride, stream);
        if (mt == 2) return launch_skinny<2, 1, 16>(a, lda, w, M, N, K, ksplit, epi, base, kparts, part_stride, stream);
        return launch_skinny<4, 1, 16>(a, lda, w, M, N, K, ksplit, epi, base, kparts, part_stride, stream);
    }
    if (mt == 1) return launch_skinny<1, 4, 4>(a, lda, w, M, N, K, ksplit, epi, base, kparts, part_stride, stream);
    if (mt == 2) return launch_skinny<2, 4, 4>(a, lda, w, M, N, K, ksplit, epi, base, kparts, part_stride, stream);
    return launch_skinny<4, 4, 4>(a, lda, w, M, N, K, ksplit, epi, base, kparts, part_stride, stream);
}

}  // namespace liyab

using namespace liyab;

// a [M <= 64, K] and w [N, K] are bfloat16. ksplit: waves per workgroup sharing K (0 = chosen
// from the shape; 1, 2, 4, 8 or 16). wide: 64 instead of 16 output features a workgroup
// (-1 = chosen from the shape). mtile: tiles of 16 rows a workgroup, 1, 2 or 4 (0 = chosen from the shape).
extern "C" int liyab_gemm_skinny(const void* a, int64_t lda, const void* w, int M, int N, int K, int ksplit, int wide,
                                 int mtile, const EpiParams* epi_in, hipStream_t stream) {
    LIYAB_REQUIRE(a && w && epi_in, "gemm: null operand");
    LIYAB_REQUIRE(M >= 0 && M <= 64 && N > 0 && K > 0, "gemm_skinny: bad sizes M=%d (at most 64) N=%d K=%d", M, N, K);
    LIYAB_REQUIRE(K % 8 == 0 && lda % 8 == 0 && lda >= K, "gemm_skinny: K %d and lda %lld must be multiples of 8", K,
                  static_cast<long long>(lda));
    LIYAB_REQUIRE((reinterpret_cast<uintptr_t>(a) & 15) == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0,
                  "gemm_skinny: operands must be 16-byte aligned");
    EpiParams epi = *epi_in;
    if (int rc = check_epilogue(epi, M, N)) return rc;
    if (M == 0) return 0;
    return skinny_dispatch(a, lda, w, M, N, K, ksplit, wide, mtile, epi, BaseSum{nullptr, 0, 0}, stream);
}

// The product's sums over `kparts` parts of K, one plane [M, N] of 32-bit sums a part:
// parts[p * part_stride + m * N + n] = sum over the p-th part of K of a[m, k] w[n, k].
// For a product with few output features and a long K: cut over K it fills the chip, and
// whoever reads the result next adds the planes up in their order (the norm kernels do).
// With `base` (n_base planes [M, N], base_stride floats apart, not overlapping `parts`), the
// first plane also takes bias[n] and base[0][m, n] + base[1][m, n] + ...: the planes together
// are then base + a . w^T + bias, the rows of a residual stream after the product was added.
// Without `base`, `bias` must be null. Every part holds at least one unit of 64 k:
// (kparts - 1) * ceil(ceil(K / 64) / kparts) * 64 < K.
extern "C" int liyab_gemm_skinny_parts(const void* a, int64_t lda, const void* w, int M, int N, int K, int kparts,
                                       int ksplit, float* parts, int64_t part_stride, const float* bias,
                                       const float* base, int n_base, int64_t base_stride, hipStream_t stream) {
    LIYAB_REQUIRE(a && w && parts, "gemm: null operand");
    LIYAB_REQUIRE(M >= 0 && M <= 64 && N > 0 && K > 0, "gemm_skinny_parts: bad sizes M=%d (at most 64) N=%d K=%d", M, N, K);
    LIYAB_REQUIRE(K % 8 == 0 && lda % 8 == 0 && lda >= K, "gemm_skinny_parts: K %d and lda %lld must be multiples of 8", K,
                  static_cast<long long>(lda));
    LIYAB_REQUIRE((reinterpret_cast<uintptr_t>(a) & 15) == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0,
                  "gemm_skinny_parts: operands must be 16-byte aligned");
    const int units = (K + 63) / 64;
    LIYAB_REQUIRE(kparts >= 1 && kparts <= 16 && (kparts - 1) * ((units + kparts - 1) / kparts) < units,
                  "gemm_skinny_parts: K = %d does not cut into %d parts of whole units of 64", K, kparts);
    LIYAB_REQUIRE(part_stride >= static_cast<int64_t>(M) * N, "gemm_skinny_parts: planes of %lld overlap", static_cast<long long>(part_stride));
    LIYAB_REQUIRE(base != nullptr || bias == nullptr, "gemm_skinny_parts: a bias needs the rows it is added to");
    if (base != nullptr) {
        LIYAB_REQUIRE(n_base >= 1 && n_base <= 16 && (n_base == 1 || base_stride >= static_cast<int64_t>(M) * N),
                      "gemm_skinny_parts: bad planes of rows to add to (%d, %lld apart)", n_base, static_cast<long long>(base_stride));
        const float* base_end = base + (n_base - 1) * base_stride + static_cast<int64_t>(M) * N;
        const float* parts_end = parts + (kparts - 1) * part_stride + static_cast<int64_t>(M) * N;
        LIYAB_REQUIRE(base_end <= parts || parts_end <= base, "gemm_skinny_parts: the rows to add to overlap the planes written");
    }
    if (M == 0) return 0;
    EpiParams epi{};
    epi.mode = kEpiNone;
    epi.out_dtype = kF32;
    epi.out = parts;
    epi.ldo = N;
    epi.bias = bias;
    // cut over K: 16 rows a workgroup (the parts cover the chip); whole: as the plain product chooses
    return skinny_dispatch(a, lda, w, M, N, K, ksplit, 0, kparts > 1 ? 1 : 0, epi, BaseSum{base, n_base, base_stride}, stream, kparts,
                           part_stride);
}

// A gated feed-forward's first product and its activation: out[m, n] = act(a[m] . w[n]) * (a[m] . w[ff + n]), a [M <= 8, K] and w [2 ff, K] bfloat16, out
// [M, ff] bfloat16, K a multiple of 64 and not of 16,384 (rings of 8 rows: 16 waves of them are the LDS a workgroup may have); act 0: silu, 1: the tanh form of gelu. The bits of liyab_gemm_skinny to 32-bit rows followed by
// liyab_glu. (8 rows, cold weights, us in two kernels and in one: 768 -> 2 x 2,048 6.8 and 5.0, 1,024 -> 2 x 2,720 7.5 and 5.5, 4,096 -> 2 x 8,064 30.0 and 26.8.)
extern "C" int liyab_gemm_skinny_glu(const void* a, int64_t lda, const void* w, int M, int ff, int K, int act, void* out, int64_t ldo, hipStream_t stream) {
    LIYAB_REQUIRE(a && w && out, "gemm_skinny_glu: null operand");
    LIYAB_REQUIRE(M >= 0 && M <= 8 && ff > 0 && K > 0 && K % kUnit == 0 && K % 16384 != 0, "gemm_skinny_glu: bad sizes M=%d (at most 8) ff=%d K=%d", M, ff, K);
    LIYAB_REQUIRE(lda % 8 == 0 && lda >= K && ldo >= ff, "gemm_skinny_glu: bad row strides %lld, %lld", static_cast<long long>(lda), static_cast<long long>(ldo));
    LIYAB_REQUIRE((reinterpret_cast<uintptr_t>(a) & 15) == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0, "gemm_skinny_glu: operands must be 16-byte aligned");
    LIYAB_REQUIRE(act == 0 || act == 1, "gemm_skinny_glu: unknown activation %d", act);
    if (M == 0) return 0;
    EpiParams epi{};
    epi.out_dtype = kBF16;
    epi.out = out;
    epi.ldo = ldo;
    // (the waves that the product alone would have: the order of its sums)
    const int units = K / kUnit, ksplit = choose_ksplit((2 * ff + 15) / 16, units, 2), pairs = (units + 1) / 2, live = ksplit < pairs ? ksplit : pairs;
    const int waves = live < 4 ? 4 : live;
    auto* pa = static_cast<const bf16_t*>(a);
    auto* pw = static_cast<const bf16_t*>(w);
#define LIYAB_GLU(EPI) launch_stream_as<bf16_t, 8, 2, 2, EPI>(pa, lda, pw, M, ff, K, ksplit, waves, epi, BaseSum{nullptr, 0, 0}, 1, K, 0, 1, stream)
    return act == 0 ? LIYAB_GLU(kEpiGluSilu) : LIYAB_GLU(kEpiGluGelu);
#undef LIYAB_GLU
}
