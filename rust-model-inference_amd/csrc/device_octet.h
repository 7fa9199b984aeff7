// One octet (eight blocks) of a Q8_0 tile against one token's staged activation: what the GEMV of single matrices and the
// kernel that walks a whole model's layers share.  A lane is (row r = lane >> 3, slice L = lane & 7).
#ifndef RMI_DEVICE_OCTET_H
#define RMI_DEVICE_OCTET_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_common.h"

namespace {

// s = f32(wd) * xs with one rounding, as _mm_mul_ps(cvtph, set1(bd)), then the block's fma.  At one token the
// product reads the f16 scale in place (h2f_times<true>: a seventh of the kernel's instructions; decode 1187 ->
// 1203 token-steps/s); with more tokens the conversion is shared and the plain multiply is the cheaper instruction.
template <bool MIX>
__device__ __forceinline__ void block_fma(float &acc, uint32_t w_bits, float xs, int wq, int xq) {
    const float s = h2f_times<MIX>(w_bits, xs);
    const int p = dot4_i8(wq, xq);
    acc = __builtin_fmaf(s, float(p), acc);
}

// The three 16-byte loads one lane issues for one octet of its row.
struct OctetRegs {
    u32x4 sc;  // 8 f16 block scales of the row (same for the 8 lanes of the row)
    u32x4 qa;  // blocks 8o..8o+3, bytes 4L..4L+3 of each
    u32x4 qb;  // blocks 8o+4..8o+7
};

__device__ __forceinline__ void load_octet(OctetRegs &g, gptr_u4 sc_ptr, gptr_u4 q_ptr, uint32_t o) {
    g.sc = sc_ptr[o * 8];
    g.qa = __builtin_nontemporal_load(q_ptr + (2 * o) * 64);  // weights are read once: do not keep them in cache
    g.qb = __builtin_nontemporal_load(q_ptr + (2 * o + 1) * 64);
}

// One token's staged operands of an octet, as a lane reads them from LDS.
struct OctetX {
    uint4 xa, xb;   // bytes 4L..4L+3 of blocks 8o..8o+3 and 8o+4..8o+7
    float4 s0, s1;  // the eight block scales
};
__device__ __forceinline__ OctetX load_octet_x(const uint4 *lds, uint32_t n_oct, uint32_t o, uint32_t L) {
    OctetX x;
    x.xa = lds[(2 * o) * 8 + L];
    x.xb = lds[(2 * o + 1) * 8 + L];
    x.s0 = reinterpret_cast<const float4 *>(lds + n_oct * 16)[2 * o];
    x.s1 = reinterpret_cast<const float4 *>(lds + n_oct * 16)[2 * o + 1];
    return x;
}
// One octet read and multiplied in place: octet_fma<1> on acc
__device__ __forceinline__ void octet_fma_one(float &acc, const OctetRegs &g, const uint4 *lds, uint32_t n_oct, uint32_t o, uint32_t L) {
    const OctetX x = load_octet_x(lds, n_oct, o, L);
    block_fma<true>(acc, g.sc.x & 0xffffu, x.s0.x, int(g.qa.x), int(x.xa.x));
    block_fma<true>(acc, g.sc.x >> 16, x.s0.y, int(g.qa.y), int(x.xa.y));
    block_fma<true>(acc, g.sc.y & 0xffffu, x.s0.z, int(g.qa.z), int(x.xa.z));
    block_fma<true>(acc, g.sc.y >> 16, x.s0.w, int(g.qa.w), int(x.xa.w));
    block_fma<true>(acc, g.sc.z & 0xffffu, x.s1.x, int(g.qb.x), int(x.xb.x));
    block_fma<true>(acc, g.sc.z >> 16, x.s1.y, int(g.qb.y), int(x.xb.y));
    block_fma<true>(acc, g.sc.w & 0xffffu, x.s1.z, int(g.qb.z), int(x.xb.z));
    block_fma<true>(acc, g.sc.w >> 16, x.s1.w, int(g.qb.w), int(x.xb.w));
}
// The NOCT octets of a tile whose weights are in registers already, one token: the LDS reads of octet o + 1 go out
// before octet o is multiplied.  A wave that has its compute unit to itself otherwise waits out an LDS round trip
// per octet (the reads of an octet and the wait for the first of them stood back to back).  Same arithmetic and
// order as octet_fma<1>.
template <int NOCT>
__device__ __forceinline__ void octets_fma_ahead(float &acc, const OctetRegs (&g)[NOCT], const uint4 *lds, uint32_t L,
                                                 uint32_t n_staged = NOCT) {  // octets staged in LDS (NOCT or more)
    OctetX x = load_octet_x(lds, n_staged, 0, L);
    float a = acc;
#pragma unroll
    for (int o = 0; o < NOCT; o++) {
        OctetX nx = x;
        if (o + 1 < NOCT) nx = load_octet_x(lds, n_staged, o + 1, L);
        // The sum passes a point that no memory access moves across: the reads of octet o + 1 stay in front of
        // the multiply-adds of octet o.  (Left to itself the compiler moves them back down to their uses.)
        asm volatile("" : "+v"(a) : : "memory");
        const OctetRegs &w = g[o];
        block_fma<true>(a, w.sc.x & 0xffffu, x.s0.x, int(w.qa.x), int(x.xa.x));
        block_fma<true>(a, w.sc.x >> 16, x.s0.y, int(w.qa.y), int(x.xa.y));
        block_fma<true>(a, w.sc.y & 0xffffu, x.s0.z, int(w.qa.z), int(x.xa.z));
        block_fma<true>(a, w.sc.y >> 16, x.s0.w, int(w.qa.w), int(x.xa.w));
        block_fma<true>(a, w.sc.z & 0xffffu, x.s1.x, int(w.qb.x), int(x.xb.x));
        block_fma<true>(a, w.sc.z >> 16, x.s1.y, int(w.qb.y), int(x.xb.y));
        block_fma<true>(a, w.sc.w & 0xffffu, x.s1.z, int(w.qb.z), int(x.xb.z));
        block_fma<true>(a, w.sc.w >> 16, x.s1.w, int(w.qb.w), int(x.xb.w));
        x = nx;
    }
    acc = a;
}

// A wave's N octets (the staged octets first .. first + N - 1) multiplied down to the two factors of every block's
// fma, for another wave to add: dst[(4 i + q) * 64] = {s, float(dot), s', float(dot')} of blocks 2q and 2q + 1 of its
// octet i (dst already points at this lane's float4).
template <int N>
__device__ __forceinline__ void octets_to_factors(const OctetRegs (&g)[N], const uint4 *lds, uint32_t n_staged,
                                                  uint32_t first, uint32_t L, float4 *dst) {
    OctetX x = load_octet_x(lds, n_staged, first, L);
#pragma unroll
    for (int i = 0; i < N; i++) {
        OctetX nx = x;
        if (i + 1 < N) nx = load_octet_x(lds, n_staged, first + i + 1, L);
        const OctetRegs &w = g[i];
        float4 *d = dst + i * 4 * 64;
        d[0] = make_float4(h2f_times<true>(w.sc.x & 0xffffu, x.s0.x), float(dot4_i8(int(w.qa.x), int(x.xa.x))),
                           h2f_times<true>(w.sc.x >> 16, x.s0.y), float(dot4_i8(int(w.qa.y), int(x.xa.y))));
        d[64] = make_float4(h2f_times<true>(w.sc.y & 0xffffu, x.s0.z), float(dot4_i8(int(w.qa.z), int(x.xa.z))),
                            h2f_times<true>(w.sc.y >> 16, x.s0.w), float(dot4_i8(int(w.qa.w), int(x.xa.w))));
        d[128] = make_float4(h2f_times<true>(w.sc.z & 0xffffu, x.s1.x), float(dot4_i8(int(w.qb.x), int(x.xb.x))),
                             h2f_times<true>(w.sc.z >> 16, x.s1.y), float(dot4_i8(int(w.qb.y), int(x.xb.y))));
        d[192] = make_float4(h2f_times<true>(w.sc.w & 0xffffu, x.s1.z), float(dot4_i8(int(w.qb.z), int(x.xb.z))),
                             h2f_times<true>(w.sc.w >> 16, x.s1.w), float(dot4_i8(int(w.qb.w), int(x.xb.w))));
        x = nx;
    }
}
// ... and the M octets' factors added to a lane's sum in block order (src points at this lane's float4 of the first)
template <int M>
__device__ __forceinline__ void factors_sum(float &acc, const float4 *src) {
    float4 f[4];
#pragma unroll
    for (int q = 0; q < 4; q++) f[q] = src[q * 64];
#pragma unroll
    for (int o = 0; o < M; o++) {
        float4 nf[4];
#pragma unroll
        for (int q = 0; q < 4; q++) nf[q] = o + 1 < M ? src[((o + 1) * 4 + q) * 64] : f[q];
        asm volatile("" : "+v"(acc) : : "memory");  // the next octet's reads stay in front of this octet's sums
#pragma unroll
        for (int q = 0; q < 4; q++) {
            acc = __builtin_fmaf(f[q].x, f[q].y, acc);
            acc = __builtin_fmaf(f[q].z, f[q].w, acc);
        }
#pragma unroll
        for (int q = 0; q < 4; q++) f[q] = nf[q];
    }
}

}  // namespace

#endif  // RMI_DEVICE_OCTET_H
