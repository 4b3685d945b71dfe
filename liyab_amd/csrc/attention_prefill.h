// What the two kernels of prompt portions' attention share: their arguments.
#pragma once

#include "common.h"

namespace liyab {

constexpr int kPrefillMaxBlocks = 2048;  // page ids of a tile's keys are kept in LDS

struct PrefillArgs {
    bf16_t* out;
    int64_t out_stride;
    const bf16_t* q;
    int64_t q_stride;
    const bf16_t *kc, *vc;
    const int* block_tables;
    int max_blocks;
    const int* work;
    float scale;
    int window, n_head, n_kv_head, hd, page_size, num_pages;
    // with SCORED
    float softcap;
    const float* bias_table;
    int max_dist;
    const float* sinks;
    int keep_first;
};

// Heads of 64 and of 128 (attention_prefill_direct.hip).
template <bool SCORED>
int launch_prefill_direct(const PrefillArgs& p, int n_tiles, int tile, int ksplit, int page_shift, hipStream_t stream);

}  // namespace liyab
