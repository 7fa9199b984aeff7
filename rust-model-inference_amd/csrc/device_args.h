// A launch's arguments, brought into the scalar cache together.
#ifndef RMI_DEVICE_ARGS_H
#define RMI_DEVICE_ARGS_H

#include <hip/hip_runtime.h>
#include <stdint.h>

// A short kernel's arguments are new to every compute unit: each 64 bytes of them are a round trip to memory of most of a
// microsecond, and the compiler, which reads an argument where it needs it, makes those trips one after the other.  This
// asks for all lines at once; what is read afterwards is in the scalar cache.  Args: the kernel's one argument, a structure,
// so that what is asked for ends where the arguments end (behind them nothing need be readable).
template <typename Args>
__device__ __forceinline__ void fetch_args() {
    constexpr uint32_t BYTES = sizeof(Args);
    static_assert(BYTES % 4 == 0, "whole words");
    constexpr uint32_t kLines = (BYTES + 63) / 64;
    const auto *p = (const __attribute__((address_space(4))) uint32_t *)__builtin_amdgcn_kernarg_segment_ptr();
    uint32_t x[kLines + 1];
#pragma unroll
    for (uint32_t i = 0; i <= kLines; i++) x[i] = p[i < kLines ? i * 16 : BYTES / 4 - 1];  // (the segment need not begin a line)
#pragma unroll
    for (uint32_t i = 0; i <= kLines; i++) asm volatile("" ::"s"(x[i]));
}

#endif  // RMI_DEVICE_ARGS_H
