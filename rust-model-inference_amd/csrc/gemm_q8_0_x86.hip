// Q8_0 products of many tokens in the x86-64 accumulation order (matmul_q8_0_vs_q8_0_avx2,
// src/ops/kernel/q8_0/avx2.rs:71-173): the bits that the GEMV of gemv_q8_0.hip gives a token, for prompt passes and
// batches of more than eight tokens (Kernel::forward_batched, src/ops/kernel/trait_.rs:78-109).
//
// The order keeps eight f32 sums per (row, token), one per 4-byte slice of a block: acc[L] = fma(wd * xd, dot4[L],
// acc[L]), block after block.  The dots come from v_mfma_f32_16x16x4_4b_f16: four independent 16 x 16 products of
// depth four, so one instruction is sixteen rows x sixteen tokens x four slices.  An int8 is exact in f16, the products
// and the sum of four of them are exact in f32, so the dot arrives as the f32 the fma takes: no conversion, and what is
// left on the vector ALU is the order's own fma and one scale product for eight of them.  Slices 2 beta and 2 beta + 1
// are the two instructions' block beta, so that a lane reads both operands of a block with one 16-byte LDS load, and
// holds all eight sums of its four rows and one token: the horizontal sum at the end crosses no lanes.
//
// What bounds it: the vector ALU, 36 instructions per 16 x 16 x 32 (32 fma, 4 scale products) = 61 ns a SIMD with four
// waves on it, 66 with two (277 / 254 TOP/s for the chip if nothing else cost anything); the matrix cores are busy half
// of that.  Converting the operands to f16 as they are staged is 5 vector instructions per 4 values, shared by the waves
// that read them.  Measured: 4096 x 1024, 512 tokens 53 -> 28 us, 151936 x 1024, 128 tokens 529 -> 220 (182 TOP/s), against
// eight tokens to a workgroup with int8 dots (4 x 4 x 4) and a conversion each, on the GEMV's kernel.
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

// A workgroup of WR x WT waves, each NR x NT tiles of sixteen rows x sixteen tokens; k in quads of four blocks through
// two LDS buffers, the next quad's bytes on their way to registers meanwhile.  One block of a buffer is [row][32 f16].
template <int NR, int NT, int WR, int WT>
struct X86Tile {
    static constexpr int BN = 16 * NR * WR, BT = 16 * NT * WT, THREADS = 64 * WR * WT;
    static constexpr int ABLK = BN * 64 + 64, BBLK = BT * 64 + 64;  // bytes of a block, off a multiple of 256
    static constexpr int LDS_BUF = 4 * (ABLK + BBLK) + 16 * (BN + BT);
};

template <int NR, int NT, int WR, int WT, int WPS>
__global__ __launch_bounds__(64 * WR * WT, WPS) void gemm_q8_0_x86_kernel(RmiGemvProblem p, uint32_t n_tokens, uint32_t grid_n,
                                                                          uint32_t grid_t, uint32_t t_fastest, uint32_t xcd_split) {
    using TL = X86Tile<NR, NT, WR, WT>;
    constexpr int BN = TL::BN, BT = TL::BT, TH = TL::THREADS;
    constexpr int PA = (BN * 8 + TH - 1) / TH, PB = (BT * 8 + TH - 1) / TH;  // 16-byte pieces a thread stages per quad
    constexpr int PS = (BT * 4 + TH - 1) / TH;
    static_assert(BN <= TH, "one thread a row for the weight scales");
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
    uint32_t a_off[PA], b_off[PB], bs_off[PS];
#pragma unroll
    for (int i = 0; i < PA; i++) {  // lane 8 r + L of a tile's pieces
        const uint32_t e = (tid + i * TH) % (BN * 8), t = (e >> 6) < last_tile ? e >> 6 : last_tile;
        a_off[i] = t * uint32_t(tile_bytes) + p.n_oct * 128 + (e & 63) * 16;
    }
    const uint32_t a_dst = ((tid % (BN * 8)) >> 3) * 64 + (tid & 7) * 8;  // piece i: TH / 8 rows on
#pragma unroll
    for (int i = 0; i < PB; i++) {  // token, half block tid & 7
        const uint32_t e = (tid + i * TH) % (BT * 8), t = (e >> 3) < last_tok ? e >> 3 : last_tok;
        b_off[i] = t * p.n_in + (tid & 1) * 16;
    }
    const uint32_t b_blk = (tid >> 1) & 3, b_dst = 4 * TL::ABLK + b_blk * TL::BBLK + ((tid % (BT * 8)) >> 3) * 64 + (tid & 1) * 32;
    const uint32_t s_row = tid < BN ? tid : BN - 1, s_tile = (s_row >> 3) < last_tile ? s_row >> 3 : last_tile;
    const uint32_t as_off = s_tile * uint32_t(tile_bytes) + (s_row & 7) * 16;
    constexpr uint32_t kScaleA = 4 * (TL::ABLK + TL::BBLK), kScaleB = kScaleA + 16 * BN;
#pragma unroll
    for (int i = 0; i < PS; i++) {
        const uint32_t e = (tid + i * TH) % (BT * 4), t = (e >> 2) < last_tok ? e >> 2 : last_tok;
        bs_off[i] = t * nb * 4;
    }
    const uint32_t bs_blk = tid & 3, bs_dst = kScaleB + (bs_blk * BT + ((tid % (BT * 4)) >> 2)) * 4;
    u32x4 ra[PA], rb[PB];
    u32x2 rsa;
    float rsb[PS];
    auto load = [&](uint32_t q) {
        // always issued (past the end the last quad again): a skipped load would make the waits wait for all of them
        q = q < n_quads ? q : n_quads - 1;
#pragma unroll
        for (int i = 0; i < PA; i++) ra[i] = *(gptr_u4)(w_base + (a_off[i] + q * 1024));
        const uint32_t bb = 4 * q + b_blk < nb ? 4 * q + b_blk : nb - 1;  // (a block past the end is not multiplied)
#pragma unroll
        for (int i = 0; i < PB; i++) rb[i] = *(gptr_u4)(x_base + (b_off[i] + bb * 32));
        rsa = *(gptr_u2)(w_base + (as_off + (q >> 1) * 128 + (q & 1) * 8));
        const uint32_t bs = 4 * q + bs_blk < nb ? 4 * q + bs_blk : nb - 1;
#pragma unroll
        for (int i = 0; i < PS; i++) rsb[i] = *(gptr_f32)(xs_base + (bs_off[i] + bs * 4));
    };
    auto park = [&](uint32_t buf) {
        uint8_t *base = lds + buf * TL::LDS_BUF;
#pragma unroll
        for (int i = 0; i < PA; i++)
#pragma unroll
            for (int b = 0; b < 4; b++) *reinterpret_cast<u32x2 *>(base + b * TL::ABLK + a_dst + i * (TH * 8)) = i8x4_to_f16x4(ra[i][b]);
#pragma unroll
        for (int i = 0; i < PB; i++)
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const u32x2 u = i8x4_to_f16x4(rb[i][2 * k]), v = i8x4_to_f16x4(rb[i][2 * k + 1]);
                *reinterpret_cast<u32x4 *>(base + b_dst + i * (TH * 8) + 16 * k) = u32x4{u[0], u[1], v[0], v[1]};
            }
        if (tid < BN) {
#pragma unroll
            for (int b = 0; b < 4; b++)
                *reinterpret_cast<float *>(base + kScaleA + (b * BN + tid) * 4) = h2f(b & 1 ? rsa[b >> 1] >> 16 : rsa[b >> 1] & 0xffffu);
        }
#pragma unroll
        for (int i = 0; i < PS; i++) *reinterpret_cast<float *>(base + bs_dst + i * TH) = rsb[i];
    };
    static_assert((BN * 8) % TH == 0 || BN * 8 < TH, "whole rounds of weight pieces");
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
        f32x4v wd[NR];
        float xd[NT];
    };
    auto read = [&](Frags &f, const uint8_t *base, int b) {
#pragma unroll
        for (int i = 0; i < NR; i++) f.a[i] = *reinterpret_cast<const u32x4 *>(base + b * TL::ABLK + (wr + i * 16 + fr) * 64 + g * 16);
#pragma unroll
        for (int j = 0; j < NT; j++) f.b[j] = *reinterpret_cast<const u32x4 *>(base + 4 * TL::ABLK + b * TL::BBLK + (wt + j * 16 + fr) * 64 + g * 16);
    };
    auto read_scales = [&](Frags &f, const uint8_t *base, int b) {
#pragma unroll
        for (int i = 0; i < NR; i++) f.wd[i] = *reinterpret_cast<const f32x4v *>(base + kScaleA + (b * BN + wr + i * 16 + g * 4) * 4);
#pragma unroll
        for (int j = 0; j < NT; j++) f.xd[j] = *reinterpret_cast<const float *>(base + kScaleB + (b * BT + wt + j * 16 + fr) * 4);
    };
    // A block's products, one ahead of the sums.  The empty statements hold that order: left to itself the compiler issues
    // every product of a quad first and spills the results, or each right in front of its sums and waits for it.  They hold
    // no instruction, so the wait states between a product and its first reader stay the compiler's own (it counts them on
    // the finished code, past such a statement; tests/test_build_checks.py pins that).
#define X86_SUMS(c) "+v"(c[0][h]), "+v"(c[0][2 + h]), "+v"(c[0][4 + h]), "+v"(c[0][6 + h]), "+v"(c[1][h]), "+v"(c[1][2 + h]), \
                    "+v"(c[1][4 + h]), "+v"(c[1][6 + h]), "+v"(c[2][h]), "+v"(c[2][2 + h]), "+v"(c[2][4 + h]), "+v"(c[2][6 + h]), \
                    "+v"(c[3][h]), "+v"(c[3][2 + h]), "+v"(c[3][4 + h]), "+v"(c[3][6 + h])
    auto product = [&](const Frags &f, int s) {
        const u32x4 a = f.a[(s >> 1) / NT], b = f.b[(s >> 1) % NT];
        const u32x2 pa = s & 1 ? u32x2{a[2], a[3]} : u32x2{a[0], a[1]}, pb = s & 1 ? u32x2{b[2], b[3]} : u32x2{b[0], b[1]};
        return __builtin_amdgcn_mfma_f32_16x16x4f16(__builtin_bit_cast(f16x4, pa), __builtin_bit_cast(f16x4, pb), zero, 0, 0, 0);
    };
    constexpr int kSteps = 2 * NR * NT;
    // d: the first product of f; returns the first one of `after`, the block behind it (nullptr: none)
    auto block = [&](const Frags &f, const Frags *after, f32x16 d) {
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
                const float sc = f.wd[i][v] * f.xd[j];
#pragma unroll
                for (int beta = 0; beta < 4; beta++) c[v][2 * beta + h] = __builtin_fmaf(sc, d[4 * beta + v], c[v][2 * beta + h]);
            }
            asm volatile("" : X86_SUMS(c));
            d = next;
        }
        return d;
    };

    load(0);
    park(0);
    load(1);
    __syncthreads();
    const uint32_t n_full = nb >> 2;
    for (uint32_t q = 0; q < n_full; q++) {
        const uint8_t *base = lds + (q & 1) * TL::LDS_BUF;
        Frags f[4];
        read(f[0], base, 0);
        f32x16 d = product(f[0], 0);
#pragma unroll
        for (int b = 0; b < 4; b++) {
            if (b < 3) read(f[b + 1], base, b + 1);
            if (NR * NT == 4 || b == 0) read_scales(f[b], base, b);  // (the largest tile has no registers for them a block ahead)
            if (NR * NT < 4 && b < 3) read_scales(f[b + 1], base, b + 1);
            d = block(f[b], b < 3 ? &f[b + 1] : nullptr, d);
        }
        park((q + 1) & 1);  // (behind the last quad: that quad again, read by nobody)
        load(q + 2);
        __syncthreads();
    }
    for (uint32_t b = 0; b < (nb & 3); b++) {  // the reference multiplies no others
        Frags f;
        read(f, lds + (n_full & 1) * TL::LDS_BUF, int(b));
        read_scales(f, lds + (n_full & 1) * TL::LDS_BUF, int(b));
        block(f, nullptr, product(f, 0));
    }

#pragma unroll
    for (int j = 0; j < NT; j++) {
        const uint32_t tok = tok0 + wt + j * 16 + fr;
        if (tok >= n_tokens) continue;
#pragma unroll
        for (int i = 0; i < NR; i++) {
            float y[4];
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const float *l = acc[i][j][v];
                y[v] = ((l[0] + l[4]) + (l[1] + l[5])) + ((l[2] + l[6]) + (l[3] + l[7]));
            }
            const uint32_t row = (p.tile0 + tile0) * 8 + wr + i * 16 + g * 4;
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
    constexpr size_t lds = 2 * TL::LDS_BUF;
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

// Which tile a product takes, or none (the GEMV's launches of up to eight tokens are faster): microseconds estimated from
// what one block of k costs a compute unit that holds w workgroups of a tile, measured on 37..151936 rows of 32..6400
// columns with 9..1000 tokens.  64 x 64: 0.43 alone, 0.71 for two (two fit); 32 x 32: 0.17, 0.25, 0.33, 0.41 for one to four
// (four fit); 64 x 16: 0.19, 0.25, 0.38 (three fit).  The GEMV: 85 TOP/s on short rows, 45 at 6400 columns, behind 4.5 us a
// launch; tokens beyond whole groups of eight are a launch of their own, which reads the weight again.
// (E.g. 4096 x 1024: 16 tokens 6.6 us there, 8.3 here; 128: 16.7 and 11.4; 512: 53 and 28.  1024 x 3072: 64 tokens 15 and
// 20 us, 512: 38 and 27.  151936 x 1024, 128 tokens: 529 and 231.)
enum X86Plan { kPlanGemv, kPlan64x64, kPlan32x32, kPlan64x16 };
X86Plan plan(uint32_t n_rows, uint32_t n_tokens, uint32_t n_in) {
    const double cus = rmi_device_cus() > 0 ? rmi_device_cus() : 1, nb = n_in / 32;
    auto estimate = [&](uint32_t bn, uint32_t bt, const double *us, int fit) {
        const double groups = double((n_rows + bn - 1) / bn) * ((n_tokens + bt - 1) / bt);
        const uint64_t w = uint64_t((groups + cus - 1) / cus);
        return 3.2 + nb * (double(w / fit) * us[fit - 1] + (w % fit ? us[w % fit - 1] : 0.0));
    };
    const uint32_t rest = n_tokens % 8;
    const double rate = 85e6 / (1.0 + (n_in > 2048 ? n_in - 2048 : 0) / 8000.0), macs = double(n_rows) * n_in;
    // (five and seven beyond whole groups cost what eight do)
    const bool whole = rest == 5 || rest == 7;
    const double gemv = 4.5 + 2.0 * macs * (n_tokens - rest) / rate +
                        (rest == 0 ? 0.0 : rest == 1 ? 2.5 + macs / 6e6 : 4.5 + (whole ? 0.04 : 0.02) * nb + macs / 12e6 + 2.0 * macs * (whole ? 8 : rest) / rate);
    const double k64[] = {0.43, 0.71}, k32[] = {0.17, 0.25, 0.33, 0.41}, k16[] = {0.19, 0.25, 0.38};
    const double t64 = estimate(64, 64, k64, 2), t32 = estimate(32, 32, k32, 4), t16 = n_tokens <= 16 ? estimate(64, 16, k16, 3) : 1e30;
    const double best = t64 < t32 ? (t64 < t16 ? t64 : t16) : (t32 < t16 ? t32 : t16);
    if (n_tokens <= 8 || gemv < best) return kPlanGemv;
    return best == t64 ? kPlan64x64 : best == t32 ? kPlan32x32 : kPlan64x16;
}

}  // namespace

bool rmi_gemm_q8_0_x86_wins(uint32_t n_rows, uint32_t n_tokens, uint32_t n_in) { return plan(n_rows, n_tokens, n_in) != kPlanGemv; }

int rmi_launch_gemm_q8_0_x86(const RmiGemvProblem &p, uint32_t n_tokens, hipStream_t s) {
    if (p.n_tiles == 0 || p.n_oct == 0 || n_tokens == 0) return RMI_HIP_OK;
    switch (plan(p.n_tiles * 8, n_tokens, p.n_in)) {
        case kPlan64x64: return launch<2, 2, 2, 2, 2>(p, n_tokens, s);
        case kPlan64x16: return launch<1, 1, 4, 1, 4>(p, n_tokens, s);
        default: return launch<1, 1, 2, 2, 4>(p, n_tokens, s);
    }
}
