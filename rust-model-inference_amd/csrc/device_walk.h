// Vectors that workgroups of one launch hand to one another, word by word (walk_qwen3.hip has the reasons).
#ifndef RMI_DEVICE_WALK_H
#define RMI_DEVICE_WALK_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_common.h"

namespace {

typedef uint64_t __attribute__((address_space(1))) *gptr_word;

// An entry of a table in HBM that the launch does not change, in scalar registers, all of it at once: what a store may change in the
// compiler's eyes it would read again, where it is used.
template <typename Entry>
__device__ __forceinline__ Entry table_entry(const Entry *entry) {
    struct Words {
        uint64_t w[sizeof(Entry) / 8];
    } e;
    static_assert(sizeof(Entry) % 8 == 0, "whole words");
    const auto *p = (const __attribute__((address_space(4))) uint64_t *)(uintptr_t)entry;
#pragma unroll
    for (uint32_t k = 0; k < sizeof(Entry) / 8; k++) e.w[k] = p[k];
#pragma unroll
    for (uint32_t k = 0; k < sizeof(Entry) / 8; k++) asm volatile("" : "+s"(e.w[k]));
    return __builtin_bit_cast(Entry, e);
}

struct WalkBound {  // of a launch's waits
    uint32_t *failed;  // set where a wait was given up
    uint32_t spins;    // how often a wait asks
};
__device__ __forceinline__ void word_store(gptr_word at, uint32_t v, uint32_t tag) {
    __hip_atomic_store(at, uint64_t(v) | (uint64_t(tag) << 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Which half of the chip this is (XCDs 0..3 and 4..7 sit on one base die each).  Every word is stored twice, and a workgroup
// reads the copy of its half: lines that are asked for on one die only.  (64 workgroups to 128 and back, 1024 words each way,
// us an exchange with 1 | 2 | 4 | 8 copies: 1.27 | 0.93 | 1.28 | 1.17; two copies by odd and even XCDs 1.26.)
__device__ __forceinline__ uint32_t die_half() {
    constexpr int kXccId = 20;  // HW_REG_XCC_ID
    return (uint32_t(__builtin_amdgcn_s_getreg((3 << 11) | kXccId)) >> 2) & 1;
}
// The N words at[i] of every lane, once all lanes' have the tag.  false: the wait was given up.
template <int N>
__device__ __forceinline__ bool words_wait(const gptr_word (&at)[N], uint32_t tag, uint32_t (&v)[N], const WalkBound &bound) {
    for (uint32_t spin = 0;; spin++) {
        uint64_t w[N];
#pragma unroll
        for (int i = 0; i < N; i++) w[i] = __hip_atomic_load(at[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        bool here = true;
#pragma unroll
        for (int i = 0; i < N; i++) {
            v[i] = uint32_t(w[i]);
            here = here && uint32_t(w[i] >> 32) == tag;
        }
        if (__all(here)) return true;
        if (spin >= bound.spins) {
            __hip_atomic_store(bound.failed, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            return false;
        }
        if ((spin & 255) == 255 && __hip_atomic_load(bound.failed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) != 0) return false;
    }
}

}  // namespace

#endif  // RMI_DEVICE_WALK_H
