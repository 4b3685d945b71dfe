// A softmax over part of a row's keys, and how two such parts become one: what the kernels that take a token's keys in a fixed order share.
#pragma once

#include "common.h"

namespace liyab {

// exponentials of scores: the fast one beside bfloat16 data, the library's beside 32-bit data
template <typename T> __device__ __forceinline__ float exp_for(float x) { return __expf(x); }
template <> __device__ __forceinline__ float exp_for<float>(float x) { return expf(x); }

struct Partial {
    float m, l;
    float acc[8];
};

// this <- merge(this, other): both rescaled to the larger maximum; this comes first. Which product of a value is rounded by itself ahead of the sum is part of a
// kernel's bits: the other's (OTHER_FIRST), or this one's; a sum's is the other's.
template <typename T, bool OTHER_FIRST>
__device__ __forceinline__ void merge_partial(Partial& a, float mo, float lo, const float* acco) {
    const float M = fmaxf(a.m, mo);
    const float wa = a.m == -INFINITY ? 0.0f : exp_for<T>(a.m - M);
    const float wb = mo == -INFINITY ? 0.0f : exp_for<T>(mo - M);
    a.l = fmaf(wa, a.l, wb * lo);
#pragma unroll
    for (int e = 0; e < 8; ++e) a.acc[e] = OTHER_FIRST ? fmaf(wa, a.acc[e], wb * acco[e]) : fmaf(wb, acco[e], wa * a.acc[e]);
    a.m = M;
}

}  // namespace liyab
