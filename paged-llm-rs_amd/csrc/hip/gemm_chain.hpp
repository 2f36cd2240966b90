// What the two chains of products (gemm_chain.hip, bfloat16; gemm_chain_f32.hip) share: how a stage of a launch leaves values for the next.
#pragma once
#include <climits>

#include "common.hpp"

typedef uint32_t cn_words4 __attribute__((ext_vector_type(4)));

#define PL_MISSING 0xffffffffu      // a word that nobody has written yet
#define CN_NOWHERE 0x7ff00000u      // an offset past every buffer's end: loads give zeros there

// Cache policies of a buffer load: device scope (sc1), and none.
struct cn_past_l2_t { static constexpr int value = 16; };
struct cn_cached_t { static constexpr int value = 0; };

__device__ __forceinline__ uint32_t cn_word(const float* p) {
    return __hip_atomic_load(reinterpret_cast<const uint32_t*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void cn_leave(void* p, uint32_t word) {
    __hip_atomic_store(static_cast<uint32_t*>(p), word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// A value is never the word that says that there is none.
__device__ __forceinline__ uint32_t cn_value(float f) {
    const uint32_t bits = __float_as_uint(f);
    return bits == PL_MISSING ? 0x7fc00000u : bits;
}

// A word of every line of the kernel's arguments, asked for at once: which of the lines a workgroup reads it learns from the first of them, and a
// second trip for another costs every workgroup some 0.5 us before it asks for its weights.
__device__ __forceinline__ void cn_touch_arguments(int bytes) {
    const __attribute__((address_space(4))) uint32_t* args = (const __attribute__((address_space(4))) uint32_t*)__builtin_amdgcn_kernarg_segment_ptr();
    uint32_t words[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) words[i] = i * 64 < bytes ? args[i * 16] : 0;
#pragma unroll
    for (int i = 0; i < 16; ++i) asm volatile("" ::"s"(words[i]));
}
