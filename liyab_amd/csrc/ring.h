// A wave's own ring in LDS for products that stream their operands: pieces of 8 rows of 64 k a load (global_load_lds, 16 bytes a lane), waited for by
// their count. A wave's loads complete in order, so no barrier is needed; what must hold is that no other load of the wave is asked for between the ring's.
#pragma once
#include "common.h"

#include <type_traits>
#include <utility>

namespace liyab {

typedef __attribute__((address_space(3))) void* lds_void_ptr;

// Where the 16-byte pieces of a ring's row sit (piece ^ swizzle), so that 16 lanes' reads of 16 rows at one piece fall into different banks.
__device__ __forceinline__ int ring_swizzle(int row) { return (row >> 1) & 7; }

// This wave's loads but the last LATER (up to 63) have arrived.
template <int LATER>
__device__ __forceinline__ void wait_loads() {
    static_assert(LATER >= 0 && LATER <= 63, "the counter of loads in flight has six bits");
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((LATER & 15) | 0x0f70 | ((LATER >> 4) << 14));
    asm volatile("" ::: "memory");
}

// f(0), f(1), ... with each number a constant.
template <int... T, typename F>
__device__ __forceinline__ void in_turn(std::integer_sequence<int, T...>, F&& f) {
    (f(std::integral_constant<int, T>{}), ...);
}

}  // namespace liyab
