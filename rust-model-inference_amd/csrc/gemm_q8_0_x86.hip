// Q8_0 products of many tokens in the x86-64 accumulation order (matmul_q8_0_vs_q8_0_avx2,
// src/ops/kernel/q8_0/avx2.rs:71-173): the bits that the GEMV of gemv_q8_0.hip gives a token, for prompt passes and
// batches of more than eight tokens (Kernel::forward_batched, src/ops/kernel/trait_.rs:78-109).
//
// The order keeps eight f32 sums per (row, token), one per 4-byte slice of a block: acc[L] = fma(wd * xd, dot4[L],
// acc[L]), block after block.  The dots come from v_mfma_f32_16x16x4_4b_f16: four independent 16 x 16 products of
// depth four, so one instruction is sixteen rows x sixteen tokens x four slices.  An int8 is exact in f16, the products
// and the sum of four of them are exact in f32, so the dot arrives as the f32 the fma takes: no conversion, and what is
// left on the vector ALU is the order's own fma.  Slices 2 beta and 2 beta + 1
// are the two instructions' block beta, so that a lane reads both operands of a block with one 16-byte LDS load, and
// holds all eight sums of its four rows and one token: the horizontal sum at the end crosses no lanes.
//
// The scale products wd * xd come from the same instruction, four outer products of sixteen rows and sixteen tokens: the weight
// scale is an f16, the token scale the reference's quantizers write is an f16 value held in an f32 (src/ops/quant/q8_0.rs:63,
// 121, 207), and the product of two f16 values is exact in f32.  (v_mfma_f32_16x16x1_4b_f32 would take any f32 scale, but f32
// products of the matrix cores and f32 sums of the vector ALU keep each other from running: 64 sums and two products 119 ns a
// wave with f16 operands, 148 with f32 ones.)  From the first quad on in which some token scale is no finite f16 value (a caller's
// own, or the quantizer's infinity for values from 8.3e6 on) a tile has scale products of the vector ALU.
//
// What bounds it: the vector ALU, 32 fma per 16 x 16 x 32 = 54 ns a SIMD with four waves on it, beside which the conversion of
// the operands to f16 as they are staged costs 5 instructions per 4 values, shared by the waves that read them: 648 vector
// instructions a quad of a wave's four tiles, with the two waves whose sums fit the registers: at 6144 x 1024, 1024 tokens they issue
// 85 % of the time, the matrix cores are busy 35 %, LDS 30 %.  us, with all scale products on the
// vector ALU | as it is | as it is, no token scale an f16 value: 64 x 64 tiles, 6144 x 1024, 1024 tokens 70.8 | 69.0 | 72.5, 151936 x
// 1024, 128 tokens 214 | 209 | 222; 32 x 32 tiles, 1024 x 3072, 512 tokens 26.1 | 25.4 | 26.6, 1024 x 2048, 512 tokens 18.5 | 18.2 |
// 19.0; 64 x 16 tiles, 20003 x 1056, 12 tokens 12.1 | 12.1 | 12.8.  (A second pass over such a tile, from memory and without
// staging, took 1085 us in the place of 73.5.)
// Eight tokens to a workgroup of the GEMV with int8 dots (4 x 4 x 4) and a conversion each: 151936 x 1024, 128 tokens 529.
#include <type_traits>

#include "rmi_internal.h"

#include "device_common.h"

namespace {

typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4v __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

// four int8 -> four f16, exact: a byte plus 128 in the low bits of 1024.0's f16 is 1152 + q
__device__ __forceinline__ u32x2 i8x4_to_f16x4(uint32_t q) {
    const uint32_t u = q ^ 0x80808080u;
    const uint32_t lo = __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u), hi = __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u);
    const f16x2 off = {_Float16(-1152.0f), _Float16(-1152.0f)};
    return u32x2{__builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, lo) + off),
                 __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, hi) + off)};
}

// A workgroup of WR x WT waves, each NR x NT tiles of sixteen rows x sixteen tokens; k in quads of four blocks through two LDS
// buffers, the next quad's bytes on their way to registers meanwhile.  One block of a buffer is [row][32 f16]; behind the blocks
// stand the quad's scales, [row][4 f16] and [token][4 f16], or, for any token scale, [block][row f32] and [block][token f32].
template <int NR, int NT, int WR, int WT>
struct X86Tile {
    static constexpr int BN = 16 * NR * WR, BT = 16 * NT * WT, THREADS = 64 * WR * WT;
    static constexpr int ABLK = BN * 64 + 64, BBLK = BT * 64 + 64;  // bytes of a block, off a multiple of 256
    static constexpr int LDS_BUF = 4 * (ABLK + BBLK) + 16 * (BN + BT);
    static constexpr int LDS = 2 * LDS_BUF + 16;  // and three flags
};

template <int NR, int NT, int WR, int WT, int WPS>
__global__ __launch_bounds__(64 * WR * WT, WPS) void gemm_q8_0_x86_kernel(RmiGemvProblem p, uint32_t n_tokens, uint32_t grid_n,
                                                                               uint32_t grid_t, uint32_t t_fastest, uint32_t xcd_split) {
    using TL = X86Tile<NR, NT, WR, WT>;
    constexpr int BN = TL::BN, BT = TL::BT, TH = TL::THREADS;
    constexpr int PA = (BN * 8 + TH - 1) / TH, PB = (BT * 8 + TH - 1) / TH;  // 16-byte pieces a thread stages per quad
    constexpr int PS = (BT * 4 + TH - 1) / TH;
    static_assert(BN <= TH, "one thread a row for the weight scales");
    static_assert(NR * NT == 1 || (NR == 2 && NT == 2), "four scale products an instruction: of four blocks or of four tiles");
    extern __shared__ uint4 lds_raw[];
    uint8_t *lds = reinterpret_cast<uint8_t *>(lds_raw);
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = uint32_t(__builtin_amdgcn_readfirstlane(int(tid >> 6)));
    const uint32_t fr = lane & 15, g = lane >> 4;
    uint32_t n_tile, t_tile;
    rmi_gemm_tile_of(blockIdx.x, grid_n, grid_t, t_fastest, xcd_split, n_tile, t_tile);
    const uint32_t tok0 = t_tile * BT, tile0 = n_tile * (BN / 8);
    const uint32_t wr = (wave % WR) * (16 * NR), wt = (wave / WR) * (16 * NT);
    const uint32_t nb = p.n_in >> 5, n_quads = (nb + 3) >> 2;
    const size_t tile_bytes = size_t(p.n_oct) * kOctetBytes;

    // ---- staging: what this thread loads of every quad (32-bit offsets from the workgroup's first tile and token)
    typedef const uint8_t __attribute__((address_space(1))) *gptr_u8;
    const gptr_u8 w_base = as_global<gptr_u8>(p.w + size_t(p.tile0 + tile0) * tile_bytes);
    const gptr_u8 x_base = as_global<gptr_u8>(p.x_q8 + size_t(tok0) * p.n_in);
    const gptr_u8 xs_base = as_global<gptr_u8>(p.x_scales + size_t(tok0) * nb);
    const uint32_t last_tile = p.n_tiles - 1 - tile0, last_tok = n_tokens - 1 - tok0;  // past them these are read again and not stored
    // weights: lane 8 r + L of a tile's pieces, each the slice L of four blocks; a wave's pieces lie in one tile
    const uint32_t a_lane = p.n_oct * 128 + (tid & 63) * 16;
    gptr_u8 a_base[PA];
#pragma unroll
    for (int i = 0; i < PA; i++) {
        const uint32_t t = wave + i * (TH / 64);
        a_base[i] = w_base + size_t(t < last_tile ? t : last_tile) * tile_bytes;
    }
    // (what follows from the thread's number in an instruction or two is made where it is used: a register less each)
    auto me = [&] {
        uint32_t t = tid;
        if (NR * NT > 1 || WT == 1) asm volatile("" : "+v"(t));
        return t;
    };
    uint32_t b_off[PB], bs_off[PS];
#pragma unroll
    for (int i = 0; i < PB; i++) {  // token, half block tid & 7
        const uint32_t e = (tid + i * TH) % (BT * 8) / 8, t = e < last_tok ? e : last_tok;
        b_off[i] = t * p.n_in + (tid & 1) * 16;
    }
    const uint32_t b_dst = 4 * TL::ABLK + (tid >> 1 & 3) * TL::BBLK + ((tid % (BT * 8)) / 8) * 64 + (tid & 1) * 32;
    const uint32_t s_row = tid % BN, s_tile = (s_row >> 3) < last_tile ? s_row >> 3 : last_tile;
    const uint32_t as_off = s_tile * uint32_t(tile_bytes) + (s_row & 7) * 16;
    constexpr uint32_t kScaleA = 4 * (TL::ABLK + TL::BBLK), kScaleB = kScaleA + 8 * BN, kScaleBAny = kScaleA + 16 * BN;
#pragma unroll
    for (int i = 0; i < PS; i++) {
        const uint32_t e = (tid + i * TH) % (BT * 4), t = (e >> 2) < last_tok ? e >> 2 : last_tok;
        bs_off[i] = t * nb * 4;
    }
    u32x4 ra[PA], rb[PB];
    u32x2 rsa;
    float rsb[PS];  // token scales, of the quad behind those in ra .. rsa
    _Float16 rsb16[PS];
    auto load_scales = [&](uint32_t q, float (&r)[PS]) {
        q = q < n_quads ? q : n_quads - 1;
        const uint32_t bs_at = 4 * q + (me() & 3), bs = bs_at < nb ? bs_at : nb - 1;
#pragma unroll
        for (int i = 0; i < PS; i++) r[i] = *(gptr_f32)(xs_base + (bs_off[i] + bs * 4));
    };
    auto load = [&](uint32_t q) {
        // always issued (past the end the last quad again): a skipped load would make the waits wait for all of them
        q = q < n_quads ? q : n_quads - 1;
#pragma unroll
        for (int i = 0; i < PA; i++) {
            uint32_t lane_off = a_lane;
            asm volatile("" : "+v"(lane_off));  // (else its sum with the base is kept, two registers a piece)
            ra[i] = *(gptr_u4)(a_base[i] + q * 1024 + lane_off);
        }
        const uint32_t t = me(), b_at = 4 * q + (t >> 1 & 3), bb = b_at < nb ? b_at : nb - 1;  // (a block past the end is not multiplied)
#pragma unroll
        for (int i = 0; i < PB; i++) rb[i] = *(gptr_u4)(x_base + (b_off[i] + bb * 32));
        rsa = *(gptr_u2)(w_base + (as_off + (q >> 1) * 128 + (q & 1) * 8));
    };
    // Whether a quad holds a token scale that is no finite f16 value is known to all waves an iteration before the quad's turn, so
    // that nobody waits for it: flag q & 1 is that of quad q, set in iteration q - 2 and read in iteration q - 1; flag 2 is quad 0's.
    uint32_t *const not_f16 = reinterpret_cast<uint32_t *>(lds + 2 * TL::LDS_BUF);
    auto take_scales = [&](const float (&r)[PS], uint32_t flag) {
#pragma unroll
        for (int i = 0; i < PS; i++) {
            rsb16[i] = _Float16(r[i]);
            // x - f32(f16(x)) is +-0 exactly when x is a finite f16 value (inf - inf and NaN are not)
            if (!(r[i] - float(rsb16[i]) == 0.0f)) not_f16[flag] = 1;
        }
    };
    auto park_scales = [&](uint8_t *base, auto any) {
        const uint32_t t = me();
        if constexpr (any.value) {
            if (t < BN) {
#pragma unroll
                for (int b = 0; b < 4; b++)
                    *reinterpret_cast<float *>(base + kScaleA + (b * BN + t) * 4) = h2f(b & 1 ? rsa[b >> 1] >> 16 : rsa[b >> 1] & 0xffffu);
            }
#pragma unroll
            for (int i = 0; i < PS; i++) *reinterpret_cast<float *>(base + kScaleBAny + ((t & 3) * BT + ((t % (BT * 4)) >> 2)) * 4 + i * TH) = rsb[i];
        } else {
            if (t < BN) *reinterpret_cast<u32x2 *>(base + kScaleA + t * 8) = rsa;
#pragma unroll
            for (int i = 0; i < PS; i++) *reinterpret_cast<_Float16 *>(base + kScaleB + (t % (BT * 4)) * 2 + i * TH * 2) = rsb16[i];
        }
    };
    const uint32_t a_dst = tid * 8;  // (kept: as it is made anew, the registers it takes keep the conversions behind the last block's sums)
    auto park = [&](uint32_t buf, auto any) {
        uint8_t *base = lds + buf * TL::LDS_BUF;
#pragma unroll
        for (int i = 0; i < PA; i++)
#pragma unroll
            for (int b = 0; b < 4; b++) *reinterpret_cast<u32x2 *>(base + a_dst + (b * TL::ABLK + i * (TH * 8))) = i8x4_to_f16x4(ra[i][b]);
#pragma unroll
        for (int i = 0; i < PB; i++)
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const u32x2 u = i8x4_to_f16x4(rb[i][2 * k]), v = i8x4_to_f16x4(rb[i][2 * k + 1]);
                *reinterpret_cast<u32x4 *>(base + b_dst + i * (TH * 8) + 16 * k) = u32x4{u[0], u[1], v[0], v[1]};
            }
        park_scales(base, any);
    };
    static_assert((BN * 8) % TH == 0, "whole rounds of weight pieces");
    static_assert((BT * 8) % TH == 0 || BT * 8 < TH, "whole rounds of token pieces");
    static_assert((BT * 4) % TH == 0 || BT * 4 < TH, "whole rounds of token scales");

    float acc[NR][NT][4][8];  // [row tile][token tile][row 4 g + v][slice]
#pragma unroll
    for (int i = 0; i < NR; i++)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int v = 0; v < 4; v++)
#pragma unroll
                for (int l = 0; l < 8; l++) acc[i][j][v][l] = 0.0f;

    f32x16 zero;
#pragma unroll
    for (int i = 0; i < 16; i++) zero[i] = 0.0f;
    struct Frags {
        u32x4 a[NR], b[NT];
    };
    const uint8_t *const read_a = lds + (wr + fr) * 64 + g * 16, *const read_b = lds + 4 * TL::ABLK + (wt + fr) * 64 + g * 16;
    auto read = [&](Frags &f, uint32_t buf, int b) {
#pragma unroll
        for (int i = 0; i < NR; i++) f.a[i] = *reinterpret_cast<const u32x4 *>(read_a + buf + (b * TL::ABLK + i * 1024));
#pragma unroll
        for (int j = 0; j < NT; j++) f.b[j] = *reinterpret_cast<const u32x4 *>(read_b + buf + (b * TL::BBLK + j * 1024));
    };
    // The scale products: outer products of sixteen rows and sixteen tokens, four of them an instruction (four tiles of a block,
    // or a tile's four blocks), in the layout of the dots.
    constexpr bool BY_TILE = NR * NT == 4;
    auto sc_a = [&](uint32_t t) { return lds + (kScaleA + wr * 8) + ((t & 15) * 8 + (BY_TILE ? (t >> 5 & 1) * 128 : (t >> 4 & 3) * 2)); };
    auto sc_b = [&](uint32_t t) { return lds + (kScaleB + wt * 8) + ((t & 15) * 8 + (BY_TILE ? (t >> 4 & 1) * 128 : (t >> 4 & 3) * 2)); };
    auto outer = [&](u32x2 a, u32x2 b) { return __builtin_amdgcn_mfma_f32_16x16x4f16(__builtin_bit_cast(f16x4, a), __builtin_bit_cast(f16x4, b), zero, 0, 0, 0); };
    // the weights' scale alone in its k slot, zero against all others (the tokens' are finite)
    auto scales_by_tile = [&](u32x2 wd, u32x2 xd, int blk) {
        return outer(u32x2{blk < 2 ? wd[0] & (blk & 1 ? 0xffff0000u : 0xffffu) : 0u, blk < 2 ? 0u : wd[1] & (blk & 1 ? 0xffff0000u : 0xffffu)}, xd);
    };
    // A block's products, one ahead of the sums.  The empty statements hold that order: left to itself the compiler issues
    // every product of a quad first and spills the results, or each right in front of its sums and waits for it.  They hold
    // no instruction, so the wait states between a product and its first reader stay the compiler's own (it counts them on
    // the finished code, past such a statement; tests/test_build_checks.py pins that).
#define X86_SUM(v, beta) "+v"(c[v][2 * (beta) + h])
#define X86_SUMS(c) X86_SUM(0, 0), X86_SUM(0, 1), X86_SUM(0, 2), X86_SUM(0, 3), X86_SUM(1, 0), X86_SUM(1, 1), X86_SUM(1, 2), X86_SUM(1, 3), \
                    X86_SUM(2, 0), X86_SUM(2, 1), X86_SUM(2, 2), X86_SUM(2, 3), X86_SUM(3, 0), X86_SUM(3, 1), X86_SUM(3, 2), X86_SUM(3, 3)
    constexpr int kSteps = 2 * NR * NT;
    auto product = [&](const Frags &f, int s) {
        const u32x4 a = f.a[(s >> 1) / NT], b = f.b[(s >> 1) % NT];
        const u32x2 pa = s & 1 ? u32x2{a[2], a[3]} : u32x2{a[0], a[1]}, pb = s & 1 ? u32x2{b[2], b[3]} : u32x2{b[0], b[1]};
        return __builtin_amdgcn_mfma_f32_16x16x4f16(__builtin_bit_cast(f16x4, pa), __builtin_bit_cast(f16x4, pb), zero, 0, 0, 0);
    };
    // d: the first product of f; returns the first one of `after`, the block behind it (nullptr: none).  scale(i, j, v): the scale
    // product of row 4 g + v and this lane's token of tile i, j
    auto block = [&](const Frags &f, const Frags *after, f32x16 d, auto scale) {
#pragma unroll
        for (int s = 0; s < kSteps; s++) {
            const int h = s & 1, i = (s >> 1) / NT, j = (s >> 1) % NT;
            auto &c = acc[i][j];
            f32x16 next = d;
            if (s + 1 < kSteps || after) {
                next = s + 1 < kSteps ? product(f, s + 1) : product(*after, 0);
                asm volatile("" : "+v"(next), X86_SUMS(c));
            }
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const float sc = scale(i, j, v);
#pragma unroll
                for (int beta = 0; beta < 4; beta++) c[v][2 * beta + h] = __builtin_fmaf(sc, d[4 * beta + v], c[v][2 * beta + h]);
            }
            asm volatile("" : X86_SUMS(c));
            d = next;
        }
        return d;
    };
    auto quad = [&](uint32_t buf) {
        Frags f[4];
        read(f[0], buf, 0);
        const uint32_t t = me();
        f32x16 sc;
        u32x2 wd, xd;
        if constexpr (BY_TILE) {
            wd = *reinterpret_cast<const u32x2 *>(sc_a(t) + buf);
            xd = *reinterpret_cast<const u32x2 *>(sc_b(t) + buf);
        } else {
            sc = outer(u32x2{*reinterpret_cast<const uint16_t *>(sc_a(t) + buf), 0u}, u32x2{*reinterpret_cast<const uint16_t *>(sc_b(t) + buf), 0u});
        }
        f32x16 d = product(f[0], 0);
#pragma unroll
        for (int b = 0; b < 4; b++) {
            if (b < 3) read(f[b + 1], buf, b + 1);
            if constexpr (BY_TILE) sc = scales_by_tile(wd, xd, b);
            d = block(f[b], b < 3 ? &f[b + 1] : nullptr, d, [&](int i, int j, int v) { return sc[4 * (BY_TILE ? i * NT + j : b) + v]; });
        }
    };

    struct Scales {
        f32x4v wd[NR];
        float xd[NT];
    };
    auto read_scales = [&](Scales &s, uint32_t buf, int b) {
        const uint32_t t = me();
#pragma unroll
        for (int i = 0; i < NR; i++) s.wd[i] = *reinterpret_cast<const f32x4v *>(lds + buf + kScaleA + (b * BN + wr + i * 16) * 4 + (t >> 4 & 3) * 16);
#pragma unroll
        for (int j = 0; j < NT; j++) s.xd[j] = *reinterpret_cast<const float *>(lds + buf + kScaleBAny + (b * BT + wt + j * 16) * 4 + (t & 15) * 4);
    };
    auto quad_any = [&](uint32_t buf) {
        Frags f[4];
        Scales s[4];
        read(f[0], buf, 0);
        f32x16 d = product(f[0], 0);
#pragma unroll
        for (int b = 0; b < 4; b++) {
            if (b < 3) read(f[b + 1], buf, b + 1);
            if (b == 0) read_scales(s[b], buf, b);
            if (b < 3) read_scales(s[b + 1], buf, b + 1);
            d = block(f[b], b < 3 ? &f[b + 1] : nullptr, d, [&](int i, int j, int v) { return s[b].wd[i][v] * s[b].xd[j]; });
        }
    };

    const uint32_t n_full = nb >> 2;
    float first[PS];
    load_scales(0, first);
    load_scales(1, rsb);
    load(0);
    if (tid < 4) not_f16[tid] = 0;
    __syncthreads();
    take_scales(first, 2);
    park(0, std::false_type());
    take_scales(rsb, 1);
    load(1);
    load_scales(2, rsb);
    __syncthreads();
    uint32_t q = 0, any = __builtin_amdgcn_readfirstlane(int(not_f16[2]));
    for (; q < n_full && !any; q++) {
        quad((q & 1) * TL::LDS_BUF);
        const uint32_t next = not_f16[(q + 1) & 1];
        park((q + 1) & 1, std::false_type());  // (behind the last quad: that quad again, read by nobody)
        take_scales(rsb, q & 1);
        load(q + 2);
        load_scales(q + 3, rsb);
        any = __builtin_amdgcn_readfirstlane(int(next));
        __syncthreads();
    }
    // A quad with a scale that is no f16 value: what is left has scale products of the vector ALU.  The quad is in its buffer, but for
    // such scales, and the next one in registers.
    if (any && q < n_quads) {
        const u32x2 wd = rsa;
        rsa = *(gptr_u2)(w_base + (as_off + (q >> 1) * 128 + (q & 1) * 8));
        load_scales(q, rsb);
        park_scales(lds + (q & 1) * TL::LDS_BUF, std::true_type());
        rsa = wd;
        load_scales(q + 1, rsb);
        __syncthreads();
    }
    for (; q < n_full; q++) {
        quad_any((q & 1) * TL::LDS_BUF);
        park((q + 1) & 1, std::true_type());
        load(q + 2);
        load_scales(q + 2, rsb);
        __syncthreads();
    }
    // the rest of a quad (the reference multiplies no others), block by block: where an instruction takes four blocks' scales they
    // are four times this one's
    const uint32_t rest = (n_full & 1) * TL::LDS_BUF;
    for (uint32_t b = 0; b < (nb & 3); b++) {
        Frags f;
        read(f, rest, int(b));
        f32x16 sc;
        if (any) {
            Scales s;
            read_scales(s, rest, int(b));
#pragma unroll
            for (int k = 0; k < 4 * NR * NT; k++) sc[k] = s.wd[k / (4 * NT)][k & 3] * s.xd[(k >> 2) % NT];
        } else {
            const uint32_t at = rest + b * 2 - (BY_TILE ? 0 : g * 2), t = me();
            sc = outer(u32x2{*reinterpret_cast<const uint16_t *>(sc_a(t) + at), 0u}, u32x2{*reinterpret_cast<const uint16_t *>(sc_b(t) + at), 0u});
        }
        block(f, nullptr, product(f, 0), [&](int i, int j, int v) { return sc[4 * (i * NT + j) + v]; });
    }

    uint32_t again = tid;
    asm volatile("" : "+v"(again));  // (what follows is not kept through the loop)
    const uint32_t lane1 = again & 63, fr1 = lane1 & 15, g1 = lane1 >> 4;
#pragma unroll
    for (int j = 0; j < NT; j++) {
        const uint32_t tok = tok0 + wt + j * 16 + fr1;
        if (tok >= n_tokens) continue;
#pragma unroll
        for (int i = 0; i < NR; i++) {
            float y[4];
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const float *l = acc[i][j][v];
                y[v] = ((l[0] + l[4]) + (l[1] + l[5])) + ((l[2] + l[6]) + (l[3] + l[7]));
            }
            const uint32_t row = (p.tile0 + tile0) * 8 + wr + i * 16 + g1 * 4;
            float *dst = p.y + size_t(tok) * p.y_stride + row;
            if (row >= p.row_start && row + 3 < p.row_end && (reinterpret_cast<uintptr_t>(dst) & 15) == 0)
                *reinterpret_cast<f32x4v *>(dst) = f32x4v{y[0], y[1], y[2], y[3]};
            else
#pragma unroll
                for (uint32_t v = 0; v < 4; v++)
                    if (row + v >= p.row_start && row + v < p.row_end) dst[v] = y[v];
        }
    }
}

template <int NR, int NT, int WR, int WT, int WPS>
int launch(const RmiGemvProblem &p, uint32_t n_tokens, hipStream_t s) {
    using TL = X86Tile<NR, NT, WR, WT>;
    constexpr size_t lds = TL::LDS;
    auto kernel = gemm_q8_0_x86_kernel<NR, NT, WR, WT, WPS>;
    if constexpr (lds > 64 * 1024) {
        static const hipError_t asked = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
        RMI_HIP_CHECK(asked);
    }
    const uint32_t gn = (p.n_tiles * 8 + TL::BN - 1) / TL::BN, gt = (n_tokens + TL::BT - 1) / TL::BT;
    const double w_bytes = double(p.n_tiles) * p.n_oct * kOctetBytes, x_bytes = double(n_tokens) * p.n_in;
    hipLaunchKernelGGL(kernel, dim3(gn * gt), dim3(TL::THREADS), lds, s, p, n_tokens, gn, gt, 1u, rmi_gemm_xcd_split(gn, gt, w_bytes, x_bytes));
    RMI_HIP_CHECK(hipGetLastError());
    return RMI_HIP_OK;
}

}  // namespace

// Which tile a product takes, or none (the GEMV's token groups are faster): microseconds estimated from what was measured on
// 300..160000 rows of 256..30720 columns with 9..1000 tokens (2600 products; the choice is 0.5 % over the best in the mean, 5 % or
// more in one of thirty-five).  A tile's launch with w workgroups a compute unit costs `block` for every block of k, by the most that a unit
// has up to four, from there on in proportion, and `group` a workgroup of a unit for what stands around its loop; within 3 % of what was
// measured.
// (E.g. 4096 x 1024: 16 tokens 5.1 us by groups, 8.0 by tiles; 64: 8.4 and 8.1; 512: 53 and 26.  1024 x 3072: 64 tokens 14.4 and
// 18.3, 512: 38 and 25.  151936 x 1024, 128 tokens: 529 and 209.  33166 x 6144, 17 tokens: 146 and 95.)
RmiX86Plan rmi_gemm_q8_0_x86_plan(uint32_t n_rows, uint32_t n_tokens, uint32_t n_in) {
    if (n_tokens <= 8 || n_rows == 0) return kX86Gemv;
    const double cus = rmi_device_cus() > 0 ? rmi_device_cus() : 1, nb = n_in / 32;
    struct Tile {
        uint32_t rows, tokens;
        double fixed, group, block[4], more, from;
    };
    auto us = [&](const Tile &t) {
        const double w = double((n_rows + t.rows - 1) / t.rows) * ((n_tokens + t.tokens - 1) / t.tokens) / cus;
        return t.fixed + t.group * w + nb * (w <= 4 ? t.block[w <= 1 ? 0 : w <= 2 ? 1 : w <= 3 ? 2 : 3] : t.more * (w + t.from));
    };
    const double t64 = us({64, 64, 3.2, 1.20, {0.428, 0.647, 1.003, 1.285}, 0.319, 0.54}),
                 t32 = us({32, 32, 2.6, 0.44, {0.173, 0.229, 0.304, 0.383}, 0.0895, 0.83}),
                 t16 = n_tokens <= 16 ? us({64, 16, 2.8, 0.57, {0.199, 0.268, 0.356, 0.487}, 0.1058, 1.06}) : 1e30;
    const double best = t64 < t32 ? (t64 < t16 ? t64 : t16) : (t32 < t16 ? t32 : t16);
    if (rmi_gemv_q8_0_groups((n_in + 255) / 256, n_rows, n_tokens).us < best) return kX86Gemv;
    return best == t64 ? kX86Tile64x64 : best == t32 ? kX86Tile32x32 : kX86Tile64x16;
}

int rmi_launch_gemm_q8_0_x86(RmiX86Plan plan, const RmiGemvProblem &p, uint32_t n_tokens, hipStream_t s) {
    if (p.n_tiles == 0 || p.n_oct == 0 || n_tokens == 0) return RMI_HIP_OK;
    switch (plan) {
        case kX86Tile64x64: return launch<2, 2, 2, 2, 2>(p, n_tokens, s);
        case kX86Tile32x32: return launch<1, 1, 2, 2, 4>(p, n_tokens, s);
        case kX86Tile64x16: return launch<1, 1, 4, 1, 4>(p, n_tokens, s);
        default: return rmi_fail(RMI_HIP_E_INVALID, "no tile size %d", int(plan));
    }
}
