// A tile of queries of prompt portions' attention, heads of 64 and of 128 (attention_prefill_direct.hip says how and why): what its kernel and the one that takes single
// tokens beside such tiles (attention_mixed.hip) share.
#pragma once
#include "attention_prefill.h"
#include "common.h"

#include <climits>

namespace liyab {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(16))) float floatx16;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((address_space(3))) void* lds_void_ptr;

// Transposing reads of LDS: 16 lanes that point at 4 keys x 16 dimensions get them back as 16 dimensions x 4 keys. Eight reads, of
// two blocks of dimensions [d], two groups of 16 keys OFF1 - OFF0 bytes apart [s], two halves of them [hh]: at[d][hh] + OFF. The wait is
// inside: the compiler's own read of this kind waits for every load from memory that goes to LDS, the next steps' keys among them.
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;
union VFrag {
    u32x2 u[2];
    bf16x8 v;
};
template <int OFF0, int OFF1>
__device__ __forceinline__ void read_values(const uint32_t (&a0)[2], const uint32_t (&a1)[2], uint32_t stage, VFrag (&f)[2][2]) {
    asm volatile(
        "ds_read_b64_tr_b16 %0, %8 offset:%12\n\t"
        "ds_read_b64_tr_b16 %1, %9 offset:%12\n\t"
        "ds_read_b64_tr_b16 %4, %10 offset:%12\n\t"
        "ds_read_b64_tr_b16 %5, %11 offset:%12\n\t"
        "ds_read_b64_tr_b16 %2, %8 offset:%13\n\t"
        "ds_read_b64_tr_b16 %3, %9 offset:%13\n\t"
        "ds_read_b64_tr_b16 %6, %10 offset:%13\n\t"
        "ds_read_b64_tr_b16 %7, %11 offset:%13\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(f[0][0].u[0]), "=&v"(f[0][0].u[1]), "=&v"(f[0][1].u[0]), "=&v"(f[0][1].u[1]), "=&v"(f[1][0].u[0]), "=&v"(f[1][0].u[1]),
          "=&v"(f[1][1].u[0]), "=&v"(f[1][1].u[1])
        : "v"(a0[0] + stage), "v"(a0[1] + stage), "v"(a1[0] + stage), "v"(a1[1] + stage), "n"(OFF0), "n"(OFF1)
        : "memory");
}

template <int HD, int QG, int KS, int NS, int STAGES>
struct DirectShape {
    static constexpr int THREADS = 64 * QG * KS, STEP = 32 * NS * KS, PIECES = HD / 8;  // 16-byte pieces a row
    static constexpr int STAGE = STEP * HD;                                        // elements of a stage's keys (as many values behind them)
    static constexpr int PARTIAL = (HD / 2) * 64 + 2 * 64;                         // floats a wave: outputs, then maximum and sum
    static constexpr int LDO = HD + 8;
    static constexpr size_t RING = size_t(STAGES) * 2 * STAGE * 2, MERGE = size_t(KS - 1) * QG * PARTIAL * 4, OUT = size_t(QG) * 32 * LDO * 2;
    static constexpr size_t BYTES = RING > MERGE ? (RING > OUT ? RING : OUT) : (MERGE > OUT ? MERGE : OUT);
};

// Where piece c of a row lies: rows are unpadded (a load fills LDS lane after lane). A 16-byte read serves 16 lanes a cycle, 16
// consecutive rows at one piece; a transposing read 32 lanes, 4 consecutive rows at 4 consecutive pieces. At 64 a head two rows
// make a round of the 64 banks: bit 1 of the row goes to the piece's highest bit (the 4 rows fall on different halves and
// halves of them), the next two bits below it (16 rows fall on 16 places); at 128 a head a row is a round, and the row's lowest two bits go on top.
template <int HD>
__device__ __forceinline__ int swizzle_of(int row) {
    return HD == 64 ? ((row >> 1) & 1) * 4 + ((row >> 2) & 3) : (row & 3) * 4 + ((row >> 2) & 3);
}

// Arguments as in attention_prefill.hip. QG x KS waves: wave (qg, ks) owns the 32 queries of group qg and, of a step's KS x NS blocks of
// 32 keys, the NS from ks NS on, a stream each; a wave's streams, then the KS partial results of a query group are merged at the end in a fixed order.
// The workgroup's LDS holds DirectShape's bytes and four a page of the block tables' width, and is declared here: as an argument, heads of 128
// took 1 to 3 % longer (us, 8 x 1,000 tokens of 12 heads 53.2 / 54.0, one of 500 of 8 12.5 / 12.9; heads of 64 even). It takes tile `tile` of the work list, head h.
template <int HD, int QG, int KS, int NS, int STAGES, bool SCORED, bool BY_LOAD>
__device__ __forceinline__ void attention_prefill_walk(PrefillArgs p, int page_shift, int h, unsigned tile) {
    extern __shared__ __attribute__((aligned(1024))) bf16_t ring[];
    typedef DirectShape<HD, QG, KS, NS, STAGES> S;
    constexpr int WK = 32 * NS, STEP = S::STEP, STAGE = S::STAGE, PIECES = S::PIECES, THREADS = S::THREADS, SLABS = HD / 16, DB = HD / 32;
    constexpr int ROWS = 64 / PIECES;             // rows a load of 1 KiB fills
    constexpr int NL = STEP / ROWS / (QG * KS);   // loads a wave of a stage's keys, and as many of its values
    static_assert(NL * ROWS * QG * KS == STEP && (STAGES - 2) * 2 * NL <= 63, "whole loads a wave, and the waits below");
    // ring: [stage][keys, values][STEP][HD]; then the partial results, then the outputs
    uint32_t* const rows_at = reinterpret_cast<uint32_t*>(reinterpret_cast<unsigned char*>(ring) + S::BYTES);  // a page's first row of this head

    const int* wk = p.work + 4 * tile;
    // (queries and positions within what the tile and the block table hold, whatever the list says)
    const int seq = wk[0], row0 = wk[1], nq = min(max(wk[3], 1), 32 * QG);
    const int pos0 = static_cast<int>(min(static_cast<int64_t>(max(wk[2], 0)), static_cast<int64_t>(p.max_blocks) * p.page_size - nq));
    const int hkv = h / (p.n_head / p.n_kv_head), window = p.window, page_size = p.page_size;
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int qg = wave % QG, ks = wave / QG;
    const int ql = lane % 32, g2 = lane / 32;
    const int* bt = p.block_tables + static_cast<int64_t>(seq) * p.max_blocks;

    const int my_q = 32 * qg + ql;
    const int qpos = pos0 + min(my_q, nq - 1);               // lanes past the tile's end repeat its last query; never stored
    const int wave_last = pos0 + min(32 * qg + 31, nq - 1);  // the wave's latest query position
    const bool wave_has = 32 * qg < nq;

    bf16x8 qf[SLABS];
    {
        const bf16_t* qrow = p.q + static_cast<int64_t>(row0 + min(my_q, nq - 1)) * p.q_stride + static_cast<int64_t>(h) * HD;
#pragma unroll
        for (int s = 0; s < SLABS; ++s) qf[s] = *reinterpret_cast<const bf16x8*>(qrow + 16 * s + 8 * g2);
    }

    const int k_hi = pos0 + nq - 1;  // last key any query of the tile sees
    int k_lo = window > 0 ? max(0, pos0 - window + 1) : 0;
    // steps ahead of the window's for positions below keep_first; none if the window's first block is not past them (one walk from 0 then)
    const int w_lo = k_lo;  // the first position the tile's windows hold
    int kept_steps = 0;
    if constexpr (SCORED) {
        if (p.keep_first > 0 && k_lo > 0) {
            kept_steps = (min(p.keep_first, k_lo) + STEP - 1) / STEP;
            if (kept_steps * STEP > (k_lo / 32) * 32) {
                kept_steps = 0;
                k_lo = 0;
            }
        }
    }
    const int kept = kept_steps > 0 ? min(p.keep_first, k_lo) : 0;  // positions the first steps hold
    const int kb0 = (k_lo / 32) * 32;                               // the window's first block
    const int kb0v = SCORED ? kb0 - kept_steps * STEP : kb0;        // where the walk's count starts
    const int units = (k_hi - kb0v) / STEP + 1;
    const int first_page = k_lo / page_size, n_pages = k_hi / page_size - first_page + 1;
    // (the host has checked that they fit; an id outside the caches' pages becomes one that exists)
    // (kept positions' pages stand ahead of the window's, as many as lie before its first page)
    const int kept_pages = SCORED && kept > 0 ? min((kept + page_size - 1) / page_size, first_page) : 0;
    auto first_row = [&](int id) {
        return static_cast<uint32_t>(min(max(id, 0), p.num_pages - 1)) * static_cast<uint32_t>(p.n_kv_head * page_size) + static_cast<uint32_t>(hkv * page_size);
    };
    for (int i = tid; i < n_pages; i += THREADS) rows_at[kept_pages + i] = first_row(bt[first_page + i]);
    if constexpr (SCORED) {
        for (int i = tid; i < kept_pages; i += THREADS) rows_at[i] = first_row(bt[i]);
    }
    // (the queries are here before the walk: inside it, a wait for them would wait for the keys ahead)
#pragma unroll
    for (int s = 0; s < SLABS; ++s) asm volatile("" : "+v"(qf[s]));
    __syncthreads();

    // A load fills ROWS consecutive rows of a stage, PIECES lanes a row. BY_LOAD: pages are a power of two and no shorter than that, so that
    // one entry of the table serves the load, its address is a scalar, and a lane only keeps to the positions inside the walk (others are masked below).
    // With other page sizes, or positions kept ahead of a window, every lane finds its own row: what lies between the kept positions and the
    // window may have been given back, and reads the window's first.
    const int my_row = lane / PIECES;
    uint32_t entry[NL];  // by load: the table's entry (the same in every lane); else this lane's row
    auto load_key = [&](int i) { return (wave * NL + i) * ROWS; };
    auto load_pos = [&](int kb, int i) { return min(max(kb + load_key(i), k_lo / ROWS * ROWS), k_hi / ROWS * ROWS); };
    auto page_of = [&](int kp) { return page_shift >= 0 ? kp >> page_shift : kp / page_size; };
    auto look_up = [&](int kb) {
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            if constexpr (BY_LOAD) {
                entry[i] = rows_at[(load_pos(kb, i) >> page_shift) - first_page];
            } else {
                const int key = load_key(i) + my_row;
                const bool early = SCORED && kb < kb0;  // a step of kept positions (the same for every thread)
                int kp = early ? min(kb - kb0v + key, kept - 1) : min(max(kb + key, k_lo), k_hi);
                if (SCORED && !early && kp < w_lo && kp >= p.keep_first) kp = w_lo;
                const int lp = page_of(kp);
                entry[i] = rows_at[SCORED && lp < first_page ? lp : kept_pages + lp - first_page] + static_cast<uint32_t>(kp - lp * page_size);
            }
        }
    };
    uint32_t piece_at[NL];  // bytes into a row
#pragma unroll
    for (int i = 0; i < NL; ++i) piece_at[i] = ((lane % PIECES) ^ swizzle_of<HD>(load_key(i) + my_row)) * 16;
    auto issue = [&](int kb, int stage) {
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            uint64_t base;
            uint32_t mine;
            if constexpr (BY_LOAD) {
                const int kp = load_pos(kb, i);
                base = static_cast<uint64_t>(static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(entry[i])) + static_cast<uint32_t>(kp & (page_size - 1))) * (2 * HD);
                mine = static_cast<uint32_t>(min(max(my_row, k_lo - kp), k_hi - kp)) * (2 * HD) + piece_at[i];
            } else {
                base = static_cast<uint64_t>(entry[i]) * (2 * HD);
                mine = piece_at[i];
            }
            bf16_t* to = ring + stage * 2 * STAGE + (wave * NL + i) * 512;
            __builtin_amdgcn_global_load_lds(reinterpret_cast<const unsigned char*>(p.kc) + base + mine, (lds_void_ptr)(to), 16, 0, 0);
            __builtin_amdgcn_global_load_lds(reinterpret_cast<const unsigned char*>(p.vc) + base + mine, (lds_void_ptr)(to + STAGE), 16, 0, 0);
        }
    };

    // Where this lane's fragments lie in a stage, in elements. Keys: row ql of a block, piece 2 sl + g2. Values: dimension 32 d +
    // ql, keys 16 s2 + 8 hh + 4 g2 + {0..3}: it points at key (lane % 16) / 4 of them, dimensions 16 ((lane % 32) / 16) + 4 (lane % 4) .. + 3 of the 32.
    int k_at[SLABS];
    uint32_t v_at[DB][2];  // (bytes, and from where LDS starts)
#pragma unroll
    for (int sl = 0; sl < SLABS; ++sl) k_at[sl] = (ks * WK + ql) * HD + ((2 * sl + g2) ^ swizzle_of<HD>(ql)) * 8;
    const uint32_t lds_start = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void_ptr)(ring)));
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
            const int key = 8 * hh + 4 * g2 + (lane % 16) / 4, dim = 32 * d + 16 * ((lane % 32) / 16) + 4 * (lane % 4);
            v_at[d][hh] = lds_start + 2 * (STAGE + (ks * WK + key) * HD + ((dim / 8) ^ swizzle_of<HD>(key)) * 8 + dim % 8);
        }

    // per stream: outputs, the reference the exponentials are taken against, and this lane's part of the sum (its own keys: the two
    // lanes of a query add theirs up at the end)
    floatx16 o_s[NS][DB];
    float m_s[NS], l_s[NS];
#pragma unroll
    for (int z = 0; z < NS; ++z) {
        m_s[z] = -INFINITY;
        l_s[z] = 0.0f;
#pragma unroll
        for (int d = 0; d < DB; ++d)
#pragma unroll
            for (int r = 0; r < 16; ++r) o_s[z][d][r] = 0.0f;
    }
    const float scale2 = (SCORED ? 1.0f : p.scale) * 1.4426950408889634f;  // log2(e): exp(x) = 2^(x log2 e)

#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s)
        if (s < units) {
            look_up(kb0v + s * STEP);
            issue(kb0v + s * STEP, s);
        }
    look_up(kb0v + (STAGES - 1) * STEP);  // (past the walk's end: its last position)
    for (int u = 0, stage = 0, next = STAGES - 1; u < units; ++u) {
        // unit u must have landed; the loads of the units after it may be in flight (a wave's loads complete in order)
        const int later = min(units - 1 - u, STAGES - 2);
        if (STAGES > 3 && later >= 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(STAGES > 3 ? 2 * 2 * NL : 0) : "memory");
        else if (STAGES > 2 && later >= 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(STAGES > 2 ? 2 * NL : 0) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        // everyone's loads of unit u are in LDS, everyone is done reading unit u - 1: its stage takes unit u + STAGES - 1
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        if (u + STAGES - 1 < units) {
            issue(kb0v + (u + STAGES - 1) * STEP, next);
            look_up(kb0v + (u + STAGES) * STEP);
        }
        const int kb_step = kb0v + u * STEP;
        const int kb = (SCORED && kb_step < kb0 ? kb_step - kb0v : kb_step) + ks * WK;  // this wave's first key
        if (wave_has && kb <= wave_last) {
            const bf16_t* at = ring + stage * 2 * STAGE;
            // S^T[key][query] = sum_d K[key][d] Q[query][d], a block of 32 keys a stream, whose products alternate
            floatx16 st[NS];
#pragma unroll
            for (int z = 0; z < NS; ++z)
#pragma unroll
                for (int r = 0; r < 16; ++r) st[z][r] = 0.0f;
            __builtin_amdgcn_s_setprio(1);
            constexpr int AHEAD = NS == 2 ? 4 : 8;  // slabs whose fragments are asked for together
#pragma unroll
            for (int s0 = 0; s0 < SLABS; s0 += AHEAD) {
                bf16x8 kf[NS][AHEAD];
#pragma unroll
                for (int sl = 0; sl < AHEAD && s0 + sl < SLABS; ++sl)
#pragma unroll
                    for (int z = 0; z < NS; ++z) kf[z][sl] = *reinterpret_cast<const bf16x8*>(at + k_at[s0 + sl] + z * 32 * HD);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int sl = 0; sl < AHEAD && s0 + sl < SLABS; ++sl)
#pragma unroll
                    for (int z = 0; z < NS; ++z) st[z] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[z][sl], qf[s0 + sl], st[z], 0, 0, 0);
            }
            const uint32_t stage_at = stage * 2 * STAGE * 2;
            VFrag vf[2][2];
            read_values<0, 16 * HD * 2>(v_at[0], v_at[1], stage_at, vf);  // (while the products run)
            __builtin_amdgcn_s_setprio(0);
            // this lane: query ql, keys kb + 32 z + 8 (r / 4) + 4 g2 + r % 4
            if constexpr (SCORED) {
#pragma unroll
                for (int z = 0; z < NS; ++z)
#pragma unroll
                    for (int r = 0; r < 16; ++r) st[z][r] *= p.scale;
                if (p.softcap > 0.0f) {
                    const float inv_cap = 1.0f / p.softcap;
#pragma unroll
                    for (int z = 0; z < NS; ++z)
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            // tanh(x) = 1 - 2 / (1 + e^(2x)), one hardware exponential and one reciprocal
                            const float e2 = __builtin_amdgcn_exp2f(2.0f * 1.4426950408889634f * st[z][r] * inv_cap);
                            st[z][r] = p.softcap * (1.0f - 2.0f * __builtin_amdgcn_rcpf(1.0f + e2));
                        }
                }
                if (p.bias_table != nullptr) {
                    // keys that lie at least max_dist behind the wave's earliest query take the table's last row throughout
                    if (pos0 + 32 * qg - (kb + WK - 1) >= p.max_dist) {
                        const float bias_far = p.bias_table[static_cast<int64_t>(p.max_dist) * p.n_head + h];
#pragma unroll
                        for (int z = 0; z < NS; ++z)
#pragma unroll
                            for (int r = 0; r < 16; ++r) st[z][r] += bias_far;
                    } else {
#pragma unroll
                        for (int z = 0; z < NS; ++z)
#pragma unroll
                            for (int r = 0; r < 16; ++r) {
                                const int kp = kb + 32 * z + 8 * (r / 4) + 4 * g2 + r % 4;
                                st[z][r] += p.bias_table[static_cast<int64_t>(min(max(qpos - kp, 0), p.max_dist)) * p.n_head + h];
                            }
                    }
                }
            }
            // keys that every query of the wave sees need no mask
            const bool whole = kb + WK - 1 <= pos0 + 32 * qg && (window <= 0 || kb > wave_last - window || (SCORED && kb + WK <= p.keep_first));
            if (!whole) {
                // key kb + 4 g2 + c, c known: a comparison and a choice a score
                const int behind = qpos - kb - 4 * g2;
#pragma unroll
                for (int z = 0; z < NS; ++z)
#pragma unroll
                    for (int r = 0; r < 16; ++r) st[z][r] = 32 * z + 8 * (r / 4) + r % 4 <= behind ? st[z][r] : -INFINITY;
                if (window > 0) {
                    const int left = behind - window, kept_to = SCORED ? p.keep_first - kb - 4 * g2 : INT_MIN;  // past the window's start, or kept
#pragma unroll
                    for (int z = 0; z < NS; ++z)
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            const int c = 32 * z + 8 * (r / 4) + r % 4;
                            if constexpr (SCORED) st[z][r] = (c > left) | (c < kept_to) ? st[z][r] : -INFINITY;
                            else st[z][r] = c > left ? st[z][r] : -INFINITY;
                        }
                }
            }
            // the reference m_s is raised only when the block's maximum passes it by more than kLag: until then exponentials may reach
            // 2^kLag, which 32-bit sums and bfloat16 products hold as well as values below 1
            constexpr float kLag = 8.0f;
            float corr[NS], ref[NS];
#pragma unroll
            for (int z = 0; z < NS; ++z) {
                float bm = st[z][0];
#pragma unroll
                for (int r = 1; r < 16; ++r) bm = fmaxf(bm, st[z][r]);
                const auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(bm), __float_as_uint(bm), false, false);  // this lane's and the lane's 32 apart
                const float b = fmaxf(__uint_as_float(both[0]), __uint_as_float(both[1])) * scale2;
                corr[z] = 1.0f;
                if (b > m_s[z] + kLag) {  // also the first block with a visible key (m_s = -inf)
                    corr[z] = m_s[z] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_s[z] - b);
                    m_s[z] = b;
                }
                ref[z] = m_s[z] == -INFINITY ? 0.0f : m_s[z];  // nothing visible yet: every score is -inf, 2^-inf = 0
            }
            bool any = false;
#pragma unroll
            for (int z = 0; z < NS; ++z) any = any || corr[z] != 1.0f;
            if (__builtin_amdgcn_ballot_w64(any) != 0) {
#pragma unroll
                for (int z = 0; z < NS; ++z)
#pragma unroll
                    for (int d = 0; d < DB; ++d)
#pragma unroll
                        for (int r = 0; r < 16; ++r) o_s[z][d][r] *= corr[z];
            }
            // exponentials, 2^(score * scale2 - reference), a stream at a time, and with them O^T[d][query] += sum_key V[key][d] P[key][query]:
            // instruction s2 contracts the keys of accumulator registers 8 s2 .. 8 s2 + 7, rows 16 s2 + 4 g2 + {0..3} and + 8
#pragma unroll
            for (int z = 0; z < NS; ++z) {
                bf16x8 pf[2];
                float bs = 0.0f;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float pr = __builtin_amdgcn_exp2f(fmaf(st[z][r], scale2, -ref[z]));  // 0 for masked keys
                    bs += pr;
                    pf[r / 8][r % 8] = static_cast<__bf16>(pr);
                }
                l_s[z] = fmaf(l_s[z], corr[z], bs);  // the reference, and so corr, is the same in both lanes of a query
#pragma unroll
                for (int d = 0; d < DB; d += 2) {
#pragma unroll
                    for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
                        for (int e = 0; e < 2; ++e) o_s[z][d + e] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[e][s2].v, pf[s2], o_s[z][d + e], 0, 0, 0);
                    // the next values: while these products run
                    if (d + 2 < DB) {
                        if (z == 0) read_values<0, 16 * HD * 2>(v_at[(d + 2) % DB], v_at[(d + 3) % DB], stage_at, vf);
                        else read_values<32 * HD * 2, 48 * HD * 2>(v_at[(d + 2) % DB], v_at[(d + 3) % DB], stage_at, vf);
                    } else if (z + 1 < NS) {
                        read_values<32 * HD * 2, 48 * HD * 2>(v_at[0], v_at[1], stage_at, vf);
                    }
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        stage = stage + 1 == STAGES ? 0 : stage + 1;
        next = next + 1 == STAGES ? 0 : next + 1;
    }
    // the streams of a wave into the first, in their order; then the two lanes of a query add up their parts of the sum
    floatx16 (&o)[DB] = o_s[0];
    float m_run = m_s[0], l_run = l_s[0];
#pragma unroll
    for (int z = 1; z < NS; ++z) {
        const float M = fmaxf(m_run, m_s[z]);
        const float wa = m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run - M);
        const float wb = m_s[z] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_s[z] - M);
        l_run = wa * l_run + wb * l_s[z];
#pragma unroll
        for (int d = 0; d < DB; ++d)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[d][r] = wa * o[d][r] + wb * o_s[z][d][r];
        m_run = M;
    }
    l_run += __shfl_xor(l_run, 32, 64);
    __syncthreads();  // nobody reads keys or values any more
    if constexpr (KS > 1) {
        // the query group's partial results, merged into wave (qg, 0) in the order of ks
        float* part = reinterpret_cast<float*>(ring);
        if (ks > 0 && wave_has) {
            float* mine = part + ((ks - 1) * QG + qg) * S::PARTIAL;
#pragma unroll
            for (int d = 0; d < DB; ++d)
#pragma unroll
                for (int r = 0; r < 16; ++r) mine[(d * 16 + r) * 64 + lane] = o[d][r];
            mine[DB * 16 * 64 + lane] = m_run;
            mine[DB * 16 * 64 + 64 + lane] = l_run;
        }
        __syncthreads();
        if (ks == 0 && wave_has) {
#pragma unroll
            for (int k2 = 1; k2 < KS; ++k2) {
                const float* other = part + ((k2 - 1) * QG + qg) * S::PARTIAL;
                const float mo = other[DB * 16 * 64 + lane], lo = other[DB * 16 * 64 + 64 + lane];
                const float M = fmaxf(m_run, mo);
                const float wa = m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run - M);
                const float wb = mo == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mo - M);
                l_run = wa * l_run + wb * lo;
#pragma unroll
                for (int d = 0; d < DB; ++d)
#pragma unroll
                    for (int r = 0; r < 16; ++r) o[d][r] = wa * o[d][r] + wb * other[(d * 16 + r) * 64 + lane];
                m_run = M;
            }
        }
        __syncthreads();  // the outputs go where the partial results lie
    }
    // o[d][r] = O^T[dim = 32 d + 8 (r / 4) + 4 g2 + r % 4][query ql]: through LDS (each wave its own rows) to rows of 16-byte pieces
    if (wave_has && ks == 0) {
        bf16_t* const rows_out = ring + qg * 32 * S::LDO;
        float inv = 1.0f / l_run;
        if constexpr (SCORED) {
            if (p.sinks != nullptr) {
                // a sink: one more term of the denominator, exp(sink) against the row's reference (both in powers of two)
                const float s2 = p.sinks[h] * 1.4426950408889634f;
                const float M = fmaxf(m_run, s2);
                const float w = m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run - M);
                inv = w / (l_run * w + __builtin_amdgcn_exp2f(s2 - M));
            }
        }
#pragma unroll
        for (int d = 0; d < DB; ++d)
#pragma unroll
            for (int r = 0; r < 16; r += 4) {
                const float v[4] = {o[d][r] * inv, o[d][r + 1] * inv, o[d][r + 2] * inv, o[d][r + 3] * inv};
                store4<bf16_t>(rows_out + ql * S::LDO + 32 * d + 2 * r + 4 * g2, v);
            }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        for (int c = lane; c < 32 * PIECES; c += 64) {
            const int qq = c / PIECES, col = (c % PIECES) * 8;
            if (32 * qg + qq < nq)
                *reinterpret_cast<u32x4*>(p.out + static_cast<int64_t>(row0 + 32 * qg + qq) * p.out_stride + static_cast<int64_t>(h) * HD + col) =
                    *reinterpret_cast<const u32x4*>(rows_out + qq * S::LDO + col);
        }
    }
}

}  // namespace liyab
