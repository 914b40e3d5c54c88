// Rows of bfloat16 operands from memory straight into LDS, for the products that stream them (gemm_skinny.hip,
// gemm_tiles.hip): global_load_lds brings 16 bytes a lane without passing through registers.
#pragma once

#include "common.h"

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

constexpr int LL_STEP = 64;      // k per step: 128 bytes of a row, one cache line
constexpr int LL_TILE = 1024;    // bytes of a load instruction: 8 rows of a step
constexpr int LL_LDS = 160 * 1024;

// 16 bytes a lane from `src` into LDS at dst + 16 * lane; counts in vmcnt.
__device__ __forceinline__ void load_to_lds(const void* src, void* dst) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                     (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

// Until at most `AT_MOST` of the wave's loads are on their way (they end in the order in which they were made).
template <int AT_MOST> __device__ __forceinline__ void wait_loads() {
    static_assert(AT_MOST >= 0 && AT_MOST < 64, "vmcnt has 6 bits");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(AT_MOST) : "memory");
}

// The same for `steps` steps of LOADS loads each behind the one that is waited for, MOST at most.
template <int LOADS, int MOST> __device__ __forceinline__ void wait_step(int steps) {
    if constexpr (MOST == 0)
        wait_loads<0>();
    else if (steps >= MOST)
        wait_loads<MOST * LOADS>();
    else
        wait_step<LOADS, MOST - 1>(steps);
}

// Place p of row r (of 16) holds piece p ^ turn(r) of the row's eight 16-byte pieces.  A 128-bit LDS read is served 16 lanes at
// a time, lanes 0-3, 12-15, 20-23 and 24-27 first: rows 0-3 and 12-15 of one lane group, 4-11 of the next, whose pieces differ.
// Rows 2j and 2j + 1 lie in the two halves of the 64 banks; this order of j keeps the eight places of a half apart for every
// such set.
__device__ __forceinline__ int turn(int r) {
    const int j = r >> 1;
    return (j & 1) | ((j >> 2) & 1) << 1 | (((j >> 1) ^ (j >> 2)) & 1) << 2;
}

static inline bool aligned16(const void* X, const void* W) { return (((uintptr_t)X | (uintptr_t)W) & 15) == 0; }

// Compute units of the current device (asked once per device).
static inline int compute_units() {
    static int known[64];
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 64) return 256;
    if (!known[device]) {
        int n = 0;
        known[device] = (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess && n > 0) ? n : 256;
    }
    return known[device];
}
