// What the attention kernels for head dimension 128 share: exact f16 products' sums in f64 over lanes and key slices.
#ifndef RMI_DEVICE_ATTN128_H
#define RMI_DEVICE_ATTN128_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_common.h"

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ half8 as_half8(const uint4 &v) { return __builtin_bit_cast(half8, v); }
__device__ __forceinline__ double quad_sum(double v) {  // (l0 + l1) + (l2 + l3) in every lane of the quad
    int lo = __double2loint(v), hi = __double2hiint(v);
    v += __hiloint2double(__builtin_amdgcn_mov_dpp(hi, 0xB1, 0xf, 0xf, true), __builtin_amdgcn_mov_dpp(lo, 0xB1, 0xf, 0xf, true));
    lo = __double2loint(v), hi = __double2hiint(v);
    v += __hiloint2double(__builtin_amdgcn_mov_dpp(hi, 0x4E, 0xf, 0xf, true), __builtin_amdgcn_mov_dpp(lo, 0x4E, 0xf, 0xf, true));
    return v;
}
// Two registers exchange lanes in one vector instruction (v_permlane32_swap: lanes 32..63 of the first with lanes
// 0..31 of the second; v_permlane16_swap: the odd rows of sixteen of the first with the even rows of the second).
// a + b afterwards is, in the lower half (the even rows), a summed over both halves (both rows of a pair), and in the
// upper half (the odd rows) b summed likewise: two values to reduce become one, without the LDS crossbar.
template <bool ROWS>
__device__ __forceinline__ double swap_add_f64(double a, double b) {
    const uint64_t ab = __builtin_bit_cast(uint64_t, a), bb = __builtin_bit_cast(uint64_t, b);
    uint64_t x, y;
    if constexpr (ROWS) {
        const auto lo = __builtin_amdgcn_permlane16_swap(uint32_t(ab), uint32_t(bb), false, false);
        const auto hi = __builtin_amdgcn_permlane16_swap(uint32_t(ab >> 32), uint32_t(bb >> 32), false, false);
        x = uint64_t(lo[0]) | (uint64_t(hi[0]) << 32);
        y = uint64_t(lo[1]) | (uint64_t(hi[1]) << 32);
    } else {
        const auto lo = __builtin_amdgcn_permlane32_swap(uint32_t(ab), uint32_t(bb), false, false);
        const auto hi = __builtin_amdgcn_permlane32_swap(uint32_t(ab >> 32), uint32_t(bb >> 32), false, false);
        x = uint64_t(lo[0]) | (uint64_t(hi[0]) << 32);
        y = uint64_t(lo[1]) | (uint64_t(hi[1]) << 32);
    }
    return __builtin_bit_cast(double, x) + __builtin_bit_cast(double, y);
}
// The eight f64 sums of a lane (dimensions 8 dg .. 8 dg + 7, dg = lane % DG_LANES) added over the wave's 64 / DG_LANES
// key slices (lanes DG_LANES apart; DG_LANES = 4, 8 or 16).  Halves, then rows, halve the values as they halve the
// lanes; what is left inside a row of sixteen goes round it by DPP.  Lane l ends with two sums, those of dimensions
// 8 dg + pv_dim_base(l) and the next one.  (f64 sums of exact terms: the order of the additions is free.)
__device__ __forceinline__ uint32_t pv_dim_base(uint32_t lane) { return 2 * ((lane >> 4) & 1) + 4 * (lane >> 5); }
template <int DG_LANES>
__device__ __forceinline__ void pv_slices_sum(const double (&acc)[8], double (&u)[2]) {
    static_assert(DG_LANES == 4 || DG_LANES == 8 || DG_LANES == 16, "slices are whole parts of a row of sixteen lanes");
    double r[4];
#pragma unroll
    for (int k = 0; k < 4; k++) r[k] = swap_add_f64<false>(acc[k], acc[k + 4]);
#pragma unroll
    for (int k = 0; k < 2; k++) {
        u[k] = swap_add_f64<true>(r[k], r[k + 2]);
        if constexpr (DG_LANES <= 8) u[k] += dpp_f64<0x128>(u[k]);  // row_ror:8
        if constexpr (DG_LANES <= 4) u[k] += dpp_f64<0x124>(u[k]);  // row_ror:4
    }
}

}  // namespace

#endif  // RMI_DEVICE_ATTN128_H
