// Attention of a prompt pass over the F16 cache, head dimension 128 (src/models/qwen3.rs:876-933): many positions of a
// head at once, with the bits that attention128_quant_kernel gives each of them alone.
//
// The reference's rounding points are kept: f16 queries, keys and values; scores as f64 sums of exact products rounded
// to f32 and scaled; the softmax numerators by the libm's expf; their sum in f32, key after key; one f32 division a
// weight, rounded to f16; the weighted values as f64 sums of exact products.  The order of the two f64 sums is free (a
// product of two f16 has 22 bits, so sums over a few thousand of them are exact but for a rounding of about 2^-53), which
// lets both be matrix products.
//
// In f64 (a workgroup of four waves takes sixteen positions of a head), v_mfma_f64_16x16x4 has the positions as its rows.
// What bounds it: the matrix cores, 64 clocks an instruction (75 TFLOP/s).
//
// In limbs (32 positions a workgroup): an f16 below 127 is a whole number of 2^-24ths in 31 bits and a sign, so four signed
// bytes hold it exactly, each worth 256 of the one before.  The product of two numbers is sixteen products of limbs, and the
// sum of many is seven int32 sums by the worth of the pair, from v_mfma_i32_16x16x64_i8: the whole sum in integers, rounded
// once where it leaves them for f64.  Sixteen int8 products take a quarter of the matrix cores' time of one in f64, and the
// weights of a block are twelve unless one of them is above 0.498.  Keys and values are split once a pass and layer, by
// attn128_limbs_kernel, which lays them out as the matrix cores take them; queries and weights by the workgroup that uses
// them.  Where a head has other keys or values (from 127 on, infinite, NaN), or a tile such queries, the tile's positions are
// done in f64.
//
// Phases of a workgroup:
//   1  scores of sixteen keys a wave and turn into a row of scratch a position, and each position's maximum;
//   2  numerators, 128 keys of all positions a turn; a lane a position adds them in order;
//   3  weights and p . v, then the quantizer: in f64 sixteen keys a wave and turn, the waves' sums meeting in LDS; in limbs
//      weights of 64 keys a wave, their limbs to LDS, and every wave 32 of the dimensions for all 256 keys.
// What bounds the second way (16 heads, a pass of 975 positions behind 1024, 112 us, where f64 took 291; 1024 positions of
// the first 1024 keys 50 us, 127): the int8 products at 2.9 POP/s in phase 1 (a third of the time; the same with the results'
// conversion or the scores' stores taken out, so the matrix cores at the clock they have under it), the f64 of the libm's
// expf and the ordered sums in phase 2 (a quarter), and the weights' division and limbs in turn with the products in phase 3.
// A prompt of 1999 tokens, 28 layers: 29.0 ms in f64, 21.5 in limbs; passes of up to 1024 positions times heads take a workgroup a position
// and head (pass_by_positions in decode_qwen3.hip).
#include "attn_prompt.h"

#include <type_traits>

#include "device_math.h"
#include "device_quant.h"

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kThreads = 256, kRows = kAttnPromptRows;  // positions of a workgroup that uses limbs; 16 of one that does not
constexpr uint32_t kTurn = 128;  // keys of a turn of phase 2

__device__ __forceinline__ double half_f64(f16x8 v, int i) { return double(float(v[i])); }
// Zeros in the place of infinities and NaN; whether there was one.
__device__ __forceinline__ bool take_out_nonfinite(f16x8 (&v)[4]) {
    uint32_t odd = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        u32x4 u = __builtin_bit_cast(u32x4, v[i]);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t lo = (u[j] & 0x7c00u) == 0x7c00u ? 0xffffu : 0u, hi = (u[j] & 0x7c000000u) == 0x7c000000u ? 0xffff0000u : 0u;
            odd |= lo | hi;
            u[j] &= ~(lo | hi);
        }
        v[i] = __builtin_bit_cast(f16x8, u);
    }
    return odd != 0;
}

struct PromptArgs {
    const uint16_t *q16, *k_cache, *v_cache;
    uint32_t step0, n_tok, kv_stride, n_head, n_head_kv, first_tile, n_tiles, half_tiles, score_stride;
    float *scratch;
    int8_t *q8;
    float *scales;
    int rounding;
    RmiAttnLimbs limbs;
};
// Which of the launch's n tiles workgroup rank i of a head takes: the longest first, and behind `half` of them the
// shortest first
__device__ __forceinline__ uint32_t prompt_tile_of(uint32_t i, uint32_t n, uint32_t half) { return i < half ? n - 1 - i : i - half; }

// ---- limbs
constexpr uint32_t kLimbTile = 1024;            // bytes of one limb of an operand of the matrix cores: sixteen a lane
constexpr uint32_t kLimbBlock = 64 * 128 * 4;   // bytes of the limbs of 64 keys (or values) of a head

// whether both halves of u are finite and below 127
__device__ __forceinline__ bool limbs_hold(uint32_t u) { return (u & 0x7fffu) < 0x57f0u && (u & 0x7fff0000u) < 0x57f00000u; }
// x = sum of limb j * 256^j; word j of the result: limb j of the four values
__device__ __forceinline__ u32x4 limbs_of(int x0, int x1, int x2, int x3) {
    constexpr uint32_t kBias = 0x808080u;  // a byte above 127 is 256 less and carries one
    const uint32_t y0 = (uint32_t(x0) + kBias) ^ kBias, y1 = (uint32_t(x1) + kBias) ^ kBias, y2 = (uint32_t(x2) + kBias) ^ kBias,
                   y3 = (uint32_t(x3) + kBias) ^ kBias;
    const uint32_t a = __builtin_amdgcn_perm(y1, y0, 0x05010400u), b = __builtin_amdgcn_perm(y3, y2, 0x05010400u);
    const uint32_t c = __builtin_amdgcn_perm(y1, y0, 0x07030602u), d = __builtin_amdgcn_perm(y3, y2, 0x07030602u);
    return u32x4{__builtin_amdgcn_perm(b, a, 0x05040100u), __builtin_amdgcn_perm(b, a, 0x07060302u), __builtin_amdgcn_perm(d, c, 0x05040100u),
                 __builtin_amdgcn_perm(d, c, 0x07060302u)};
}
__device__ __forceinline__ int in_units(_Float16 h) { return int(float(h) * 0x1p24f); }
// limb j of sixteen values: l[j]
__device__ __forceinline__ void limbs_of16(const _Float16 (&h)[16], u32x4 (&l)[4]) {
#pragma unroll
    for (int w = 0; w < 4; w++) {
        const u32x4 v = limbs_of(in_units(h[4 * w]), in_units(h[4 * w + 1]), in_units(h[4 * w + 2]), in_units(h[4 * w + 3]));
#pragma unroll
        for (int j = 0; j < 4; j++) l[j][w] = v[j];
    }
}
__device__ __forceinline__ i32x4 mma_i8(u32x4 a, u32x4 b, i32x4 c) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, a), __builtin_bit_cast(i32x4, b), c, 0, 0, 0);
}

// Workgroup (block, head, 0): keys 64 block .. + 63 of the head; (block, head, 1): their values.  Keys behind n_keys are
// zeros.  Laid out as operands: keys [four tiles of sixteen][half of the dimensions][limb], lane (c16, g) of each the
// dimensions 16 g .. + 15 of the half of key c16; values [eight tiles of sixteen dimensions][limb], lane (c16, g) the keys
// 16 g .. + 15 of dimension c16.  What bounds it: the cache rows read and twice their bytes written.
__global__ __launch_bounds__(kThreads) void attn128_limbs_kernel(const uint16_t *__restrict__ k_cache, const uint16_t *__restrict__ v_cache,
                                                                 uint32_t n_keys, uint32_t kv_stride, RmiAttnLimbs limbs) {
    constexpr uint32_t kRowBytes = 130 * 2;  // from key to key: sixteen keys on are sixteen banks on
    __shared__ __attribute__((aligned(16))) uint8_t rows[64 * kRowBytes];
    const uint32_t tid = threadIdx.x, block = blockIdx.x, kvh = blockIdx.y, n_kv = gridDim.y, what = blockIdx.z;
    uint8_t *dst = (what ? limbs.v : limbs.k) + (size_t(kvh) * limbs.blocks + block) * kLimbBlock;
    const uint16_t *src = (what ? v_cache : k_cache) + size_t(kvh) * 128;
    bool wide = false;
#pragma unroll
    for (uint32_t i = 0; i < 2; i++) {  // sixteen dimensions of a key
        const uint32_t e = tid + i * kThreads, tile = e >> 7, half = (e >> 6) & 1, lane = e & 63;
        const uint32_t key = block * 64 + tile * 16 + (lane & 15), d0 = half * 64 + (lane >> 4) * 16;
        u32x4 u[2] = {u32x4{0, 0, 0, 0}, u32x4{0, 0, 0, 0}};
        if (key < n_keys) {
            const u32x4 *p = reinterpret_cast<const u32x4 *>(src + size_t(key) * kv_stride + d0);
            u[0] = p[0];
            u[1] = p[1];
        }
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int k = 0; k < 4; k++) wide |= !limbs_hold(u[j][k]);
        if (what == 0) {
            _Float16 h[16];
#pragma unroll
            for (int j = 0; j < 16; j++) h[j] = __builtin_bit_cast(f16x8, u[j >> 3])[j & 7];
            u32x4 l[4];
            limbs_of16(h, l);
#pragma unroll
            for (int j = 0; j < 4; j++) *reinterpret_cast<u32x4 *>(dst + (((tile * 2 + half) * 4 + j) * kLimbTile + lane * 16)) = l[j];
        } else {
#pragma unroll
            for (int k = 0; k < 8; k++)
                *reinterpret_cast<uint32_t *>(rows + (tile * 16 + (lane & 15)) * kRowBytes + d0 * 2 + k * 4) = u[k >> 2][k & 3];
        }
    }
    wide = __syncthreads_or(wide);
    if (tid == 0) limbs.wide[(what * n_kv + kvh) * limbs.blocks + block] = wide ? 1u : 0u;
    if (what == 0) return;
#pragma unroll
    for (uint32_t i = 0; i < 2; i++) {  // sixteen keys of a dimension
        const uint32_t e = tid + i * kThreads, tile = e >> 6, lane = e & 63;
        _Float16 h[16];
#pragma unroll
        for (uint32_t j = 0; j < 16; j++) h[j] = *reinterpret_cast<const _Float16 *>(rows + ((lane >> 4) * 16 + j) * kRowBytes + (tile * 16 + (lane & 15)) * 2);
        u32x4 l[4];
        limbs_of16(h, l);
#pragma unroll
        for (int j = 0; j < 4; j++) *reinterpret_cast<u32x4 *>(dst + ((tile * 4 + j) * kLimbTile + lane * 16)) = l[j];
    }
}

// ---- the pass
constexpr uint32_t kSuper = 4;  // blocks of 64 keys whose weights are in LDS at once
template <uint32_t ROWS>
struct PromptLds {
    union {
        u32x4 q[4][4][64];                     // 1: [positions' half * 2 + dimensions' half][limb][lane]
        float turn[2][ROWS][kTurn + 4];        // 2; four lanes' 16-byte reads on different banks
        u32x4 p[ROWS / 16][kSuper][2][4][64];  // 3: [buffer][block][positions' half][limb][lane]
        double part[3][16][128];               // 3 in f64: three waves' sums
        float out[ROWS][128 + 4];
    };
    float row_max[4][ROWS], row_sum[ROWS];
    uint64_t exp_tab[32];
    uint32_t top[2][kSuper];  // whether any weight of a block has a fourth limb
};

// What the f64 products take and give: lane (c16, g) has key (of sixteen) c16 and position 4 i + g of the half in register i
// of a score, position 4 i + g and dimension 8 c16 + j in register i of sum j.

// Phase 1 in f64: lane (c16, g) gives the matrix cores dimensions (4 c + g) * 8 .. + 7, c = 0..3, of position (as A) or key
// (as B) c16: sixteen bytes a load, four lanes of a key 64 consecutive bytes
template <uint32_t ROWS>
__device__ __forceinline__ void wide_scores(const PromptArgs &a, PromptLds<ROWS> &l, uint32_t head, uint32_t kvh, uint32_t t0, uint32_t rows, float *s_row0) {
    constexpr uint32_t RT = ROWS / 16;
    const uint32_t lane = threadIdx.x & 63, wave = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)));
    const uint32_t c16 = lane & 15, g = lane >> 4, n_keys = a.step0 + t0 + rows, key_tiles = (n_keys + 15) / 16;
    f16x8 qh[RT][4];
#pragma unroll
    for (uint32_t rt = 0; rt < RT; rt++) {
        const uint32_t t = t0 + (rt * 16 + c16 < rows ? rt * 16 + c16 : rows - 1);
        const uint16_t *src = a.q16 + (size_t(t) * a.n_head + head) * 128 + g * 8;
#pragma unroll
        for (int c = 0; c < 4; c++) qh[rt][c] = *reinterpret_cast<const f16x8 *>(src + c * 32);
    }
    const uint16_t *kbase = a.k_cache + size_t(kvh) * 128 + g * 8;
    auto load_keys = [&](f16x8 (&kk)[4], uint32_t kt) {  // (past the last position: that one again, masked below)
        const uint32_t key = kt * 16 + c16 < n_keys ? kt * 16 + c16 : n_keys - 1;
        const uint16_t *src = kbase + size_t(key) * a.kv_stride;
#pragma unroll
        for (int c = 0; c < 4; c++) kk[c] = *reinterpret_cast<const f16x8 *>(src + c * 32);
    };
    const float kq_scale = 1.0f / sqrtf(128.0f);  // two f32 roundings, as the reference computes it
    float my_max[RT][4];
#pragma unroll
    for (uint32_t rt = 0; rt < RT; rt++)
#pragma unroll
        for (int i = 0; i < 4; i++) my_max[rt][i] = -INFINITY;
    f16x8 kk[4], kn[4];
    load_keys(kk, wave);
    for (uint32_t kt = wave; kt < key_tiles; kt += 4) {
        load_keys(kn, kt + 4);
        f64x4 s[RT][2];
#pragma unroll
        for (uint32_t rt = 0; rt < RT; rt++) s[rt][0] = s[rt][1] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const double k = half_f64(kk[c], j);
#pragma unroll
                for (uint32_t rt = 0; rt < RT; rt++) s[rt][j & 1] = __builtin_amdgcn_mfma_f64_16x16x4f64(half_f64(qh[rt][c], j), k, s[rt][j & 1], 0, 0, 0);
            }
        const uint32_t key = kt * 16 + c16;
#pragma unroll
        for (uint32_t rt = 0; rt < RT; rt++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t r = rt * 16 + 4 * i + g;
                const float sc = float(s[rt][0][i] + s[rt][1][i]) * kq_scale;
                if (key <= a.step0 + t0 + r) my_max[rt][i] = fmaxf(my_max[rt][i], sc);
                s_row0[size_t(r) * a.score_stride + key] = sc;
            }
#pragma unroll
        for (int c = 0; c < 4; c++) kk[c] = kn[c];
    }
#pragma unroll
    for (uint32_t rt = 0; rt < RT; rt++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float m = my_max[rt][i];
            m = fmaxf(m, dpp_f32<kDppQuadXor1>(m));
            m = fmaxf(m, dpp_f32<kDppQuadXor2>(m));
            m = fmaxf(m, dpp_f32<kDppRowHalfMirror>(m));
            m = fmaxf(m, dpp_f32<kDppRowMirror>(m));
            if (c16 == 0) l.row_max[wave][rt * 16 + 4 * i + g] = m;
        }
}

// Phase 3 in f64.  Lane (c16, g): weights of position c16 and keys 4 g .. 4 g + 3 of the sixteen (as A); dimensions
// 8 c16 .. + 7 of the same keys (as B), so that product j's columns are the dimensions 8 c16 + j.  A key behind a position
// has weight zero there, which hides its value as long as that is finite (0 x inf is NaN, which the quantizer drops): of the
// few keys that some positions of the tile see and others do not, other values are taken out and counted afterwards.
template <uint32_t ROWS>
__device__ __forceinline__ void wide_values(const PromptArgs &a, PromptLds<ROWS> &l, uint32_t kvh, uint32_t t0, uint32_t rows, const float *s_row0) {
    constexpr uint32_t RT = ROWS / 16;
    const uint32_t lane = threadIdx.x & 63, wave = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)));
    const uint32_t c16 = lane & 15, g = lane >> 4, n_keys = a.step0 + t0 + rows, key_tiles = (n_keys + 15) / 16;
    const uint16_t *vbase = a.v_cache + size_t(kvh) * 128 + c16 * 8;
    f64x4 acc[RT][8];
#pragma unroll
    for (uint32_t rt = 0; rt < RT; rt++)
#pragma unroll
        for (int j = 0; j < 8; j++) acc[rt][j] = f64x4{0.0, 0.0, 0.0, 0.0};
    float total[RT];
#pragma unroll
    for (uint32_t rt = 0; rt < RT; rt++) total[rt] = l.row_sum[rt * 16 + c16];
    auto weight = [&](float ev, uint32_t rt) { return double(h2f(rmi_f2h(total[rt] > 0.0f ? ev / total[rt] : ev))); };
    const float *wsrc = s_row0 + size_t(c16) * a.score_stride + 4 * g;
    auto load_values = [&](f16x8 (&vv)[4], float4 (&e)[RT], uint32_t kt) {
        kt = kt < key_tiles ? kt : key_tiles - 1;
#pragma unroll
        for (uint32_t rt = 0; rt < RT; rt++) e[rt] = *reinterpret_cast<const float4 *>(wsrc + size_t(rt) * 16 * a.score_stride + kt * 16);
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) {
            const uint32_t key = kt * 16 + 4 * g + i < n_keys ? kt * 16 + 4 * g + i : n_keys - 1;
            vv[i] = *reinterpret_cast<const f16x8 *>(vbase + size_t(key) * a.kv_stride);
        }
    };
    bool odd = false;
    f16x8 vv[4], vn[4];
    float4 e[RT], en[RT];
    load_values(vv, e, wave);
    for (uint32_t kt = wave; kt < key_tiles; kt += 4) {
        load_values(vn, en, kt + 4);
        if (kt * 16 + 15 > a.step0 + t0) odd |= take_out_nonfinite(vv);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            double w[RT];
#pragma unroll
            for (uint32_t rt = 0; rt < RT; rt++) w[rt] = weight(i == 0 ? e[rt].x : i == 1 ? e[rt].y : i == 2 ? e[rt].z : e[rt].w, rt);
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const double v = half_f64(vv[i], j);
#pragma unroll
                for (uint32_t rt = 0; rt < RT; rt++) acc[rt][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(w[rt], v, acc[rt][j], 0, 0, 0);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; i++) vv[i] = vn[i];
#pragma unroll
        for (uint32_t rt = 0; rt < RT; rt++) e[rt] = en[rt];
    }
    if (__any(odd))  // what was taken out, one position after the other, without the values behind it
        for (uint32_t kt = wave; kt < key_tiles; kt += 4) {
            if (kt * 16 + 15 <= a.step0 + t0) continue;
#pragma unroll 1
            for (uint32_t r = 0; r < rows; r++)
#pragma unroll 1
                for (uint32_t i = 0; i < 4; i++) {
                    const uint32_t key = kt * 16 + 4 * g + i, there = key < n_keys ? key : n_keys - 1;
                    const double w = weight(wsrc[size_t(r & 16) * a.score_stride + kt * 16 + i], RT > 1 && r >= 16);
                    const f16x8 v = *reinterpret_cast<const f16x8 *>(vbase + size_t(there) * a.kv_stride);
#pragma unroll
                    for (int j = 0; j < 8; j++) {
                        const bool finite = fabsf(float(v[j])) <= 65504.0f;
                        const f64x4 o = __builtin_amdgcn_mfma_f64_16x16x4f64(w, finite || key > a.step0 + t0 + r ? 0.0 : half_f64(v, j), f64x4{0.0, 0.0, 0.0, 0.0}, 0, 0, 0);
#pragma unroll
                        for (uint32_t rt = 0; rt < RT; rt++)
#pragma unroll
                            for (uint32_t q = 0; q < 4; q++) acc[rt][j][q] += rt * 16 + 4 * q + g == r ? o[q] : 0.0;
                    }
                }
        }
    float o[RT][4][8];  // the first wave's
#pragma unroll
    for (uint32_t rt = 0; rt < RT; rt++) {
        if (wave > 0) {
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 8; j++) l.part[wave - 1][4 * i + g][8 * c16 + j] = acc[rt][j][i];
        }
        __syncthreads();
        if (wave == 0) {
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const uint32_t r = 4 * i + g, d = 8 * c16 + j;
                    o[rt][i][j] = float(((acc[rt][j][i] + l.part[0][r][d]) + l.part[1][r][d]) + l.part[2][r][d]);
                }
        }
        __syncthreads();
    }
    if (wave == 0) {
#pragma unroll
        for (uint32_t rt = 0; rt < RT; rt++)
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 8; j++) l.out[rt * 16 + 4 * i + g][8 * c16 + j] = o[rt][i][j];
    }
}

// Phase 1 in limbs.  The result of a product has position c16 of the half and keys 4 g .. 4 g + 3 in its four registers.
__device__ __forceinline__ void limb_scores(const PromptArgs &a, PromptLds<kRows> &l, uint32_t kvh, uint32_t t0, uint32_t rows, float *s_row0) {
    const uint32_t lane = threadIdx.x & 63, wave = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)));
    const uint32_t c16 = lane & 15, g = lane >> 4, n_keys = a.step0 + t0 + rows, key_tiles = (n_keys + 15) / 16;
    u32x4 q[2][2][4];
#pragma unroll
    for (int rt = 0; rt < 2; rt++)
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
            for (int j = 0; j < 4; j++) q[rt][c][j] = l.q[rt * 2 + c][j][lane];
    const uint8_t *kbase = a.limbs.k + size_t(kvh) * a.limbs.blocks * kLimbBlock + lane * 16;
    auto load_keys = [&](u32x4 (&kk)[2][4], uint32_t kt) {  // (past the last tile: that one again, not used)
        kt = kt < key_tiles ? kt : key_tiles - 1;
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
            for (int j = 0; j < 4; j++) kk[c][j] = *reinterpret_cast<const u32x4 *>(kbase + (size_t(kt) * 8 + c * 4 + j) * kLimbTile);
    };
    // two f32 roundings, as the reference computes it, and the unit of a product of limbs: a power of two, exact
    const float scale = 1.0f / sqrtf(128.0f) * 0x1p-48f;
    float my_max[2] = {-INFINITY, -INFINITY};
    auto tile_scores = [&](const u32x4 (&kk)[2][4], uint32_t kt) {
        const uint32_t key = kt * 16 + 4 * g;
        const bool behind = kt * 16 + 15 > a.step0 + t0;  // keys that a position does not see among them
#pragma unroll
        for (int rt = 0; rt < 2; rt++) {
            i32x4 s[7];
#pragma unroll
            for (int j = 0; j < 7; j++) s[j] = i32x4{0, 0, 0, 0};
#pragma unroll
            for (int c = 0; c < 2; c++)
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int j = 0; j < 4; j++) s[i + j] = mma_i8(kk[c][j], q[rt][c][i], s[i + j]);
            f32x4 sc;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                // |s[0]| <= 2^21, |s[1]| <= 2^22, |s[2]|, |s[4]| <= 3 2^21, |s[3]| <= 2^23, |s[5]| <= 2^22, |s[6]| <= 2^21:
                // the sums of two fit an int32, what is below f64's one rounding is exact
                const int s12 = s[1][i] + (s[2][i] << 8), s34 = s[3][i] + (s[4][i] << 8), s56 = s[5][i] + (s[6][i] << 8);
                const double lo = __builtin_fma(double(s12), 0x1p8, double(s[0][i])), hi = __builtin_fma(double(s56), 0x1p16, double(s34));
                sc[i] = float(__builtin_fma(hi, 0x1p24, lo)) * scale;
            }
            const uint32_t r = rt * 16 + c16;
            *reinterpret_cast<f32x4 *>(s_row0 + (size_t(r) * a.score_stride + key)) = sc;
            if (behind)
#pragma unroll
                for (uint32_t i = 0; i < 4; i++) sc[i] = key + i <= a.step0 + t0 + r ? sc[i] : -INFINITY;
            my_max[rt] = fmaxf(fmaxf(fmaxf(my_max[rt], sc[0]), fmaxf(sc[1], sc[2])), sc[3]);
        }
    };
    u32x4 k0[2][4], k1[2][4];
    load_keys(k0, wave);
    for (uint32_t kt = wave; kt < key_tiles; kt += 8) {
        load_keys(k1, kt + 4);
        tile_scores(k0, kt);
        load_keys(k0, kt + 8);
        if (kt + 4 < key_tiles) tile_scores(k1, kt + 4);
    }
#pragma unroll
    for (int rt = 0; rt < 2; rt++) {
        const float m = fmaxf(my_max[rt], __shfl_xor(my_max[rt], 16)), m2 = fmaxf(m, __shfl_xor(m, 32));
        if (g == 0) l.row_max[wave][rt * 16 + c16] = m2;
    }
}
// Phase 3 in limbs.  Numerators behind a position are zeros, and so are its weights there.
__device__ __forceinline__ void limb_values(const PromptArgs &a, PromptLds<kRows> &l, uint32_t kvh, uint32_t t0, uint32_t rows, const float *s_row0) {
    const uint32_t lane = threadIdx.x & 63, wave = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)));
    const uint32_t c16 = lane & 15, g = lane >> 4, n_keys = a.step0 + t0 + rows, n_blocks = (n_keys + 63) / 64;
    i32x4 acc[2][2][7];  // [positions' half][sixteen dimensions][worth]
#pragma unroll
    for (int rt = 0; rt < 2; rt++)
#pragma unroll
        for (int dt = 0; dt < 2; dt++)
#pragma unroll
            for (int j = 0; j < 7; j++) acc[rt][dt][j] = i32x4{0, 0, 0, 0};
    {
        // Numerators and sum are normal f32 (the largest numerator is one), so the f64 product with the reciprocal, off by
        // at most 2^-52, rounds to the f32 quotient: that lies 2^-49 or more from the middle of two neighbours.  (Quotients
        // below f32's normal range are zeros in f16 either way.)
        const double inv[2] = {1.0 / double(l.row_sum[c16]), 1.0 / double(l.row_sum[16 + c16])};
        const float *wsrc = s_row0 + size_t(c16) * a.score_stride + g * 16;
        // of this wave's block of super-block sb
        auto load_numerators = [&](float4 (&e)[2][4], uint32_t sb) {
            const uint32_t b = sb * kSuper + wave < n_blocks ? sb * kSuper + wave : n_blocks - 1;
#pragma unroll
            for (int rt = 0; rt < 2; rt++)
#pragma unroll
                for (int j = 0; j < 4; j++) e[rt][j] = *reinterpret_cast<const float4 *>(wsrc + size_t(rt) * 16 * a.score_stride + b * 64 + j * 4);
        };
        auto park_weights = [&](const float4 (&e)[2][4], uint32_t buf) {
            uint32_t top = 0;
#pragma unroll
            for (int rt = 0; rt < 2; rt++) {
                _Float16 h[16];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float ev[4] = {e[rt][j].x, e[rt][j].y, e[rt][j].z, e[rt][j].w};
#pragma unroll
                    for (int k = 0; k < 4; k++) h[4 * j + k] = __builtin_bit_cast(_Float16, rmi_f2h(float(double(ev[k]) * inv[rt])));
                }
                u32x4 pl[4];
                limbs_of16(h, pl);
#pragma unroll
                for (int j = 0; j < 4; j++) l.p[buf][wave][rt][j][lane] = pl[j];
                top |= pl[3][0] | pl[3][1] | pl[3][2] | pl[3][3];
            }
            const bool any = __any(top != 0);
            if (lane == 0) l.top[buf][wave] = any ? 1u : 0u;
        };
        const uint8_t *vbase = a.limbs.v + size_t(kvh) * a.limbs.blocks * kLimbBlock + wave * 2 * 4 * kLimbTile + lane * 16;
        auto load_values = [&](u32x4 (&vv)[2][4], uint32_t b) {
            b = b < n_blocks ? b : n_blocks - 1;
#pragma unroll
            for (int dt = 0; dt < 2; dt++)
#pragma unroll
                for (int j = 0; j < 4; j++) vv[dt][j] = *reinterpret_cast<const u32x4 *>(vbase + size_t(b) * kLimbBlock + (dt * 4 + j) * kLimbTile);
        };
        const uint32_t n_super = (n_blocks + kSuper - 1) / kSuper;
        float4 e[2][4];
        u32x4 vv[2][4];
        load_numerators(e, 0);
        load_values(vv, 0);
        park_weights(e, 0);
        __syncthreads();
        for (uint32_t sb = 0; sb < n_super; sb++) {
            const uint32_t buf = sb & 1;
#pragma unroll 1
            for (uint32_t i = 0; i < kSuper; i++) {
                const uint32_t b = sb * kSuper + i;
                if (b >= n_blocks) break;
                u32x4 vn[2][4];
                load_values(vn, b + 1);
                auto multiply = [&](int from, int to) {
#pragma unroll
                    for (int rt = 0; rt < 2; rt++)
#pragma unroll
                        for (int i2 = from; i2 < to; i2++) {
                            const u32x4 p = l.p[buf][i][rt][i2][lane];
#pragma unroll
                            for (int dt = 0; dt < 2; dt++)
#pragma unroll
                                for (int j = 0; j < 4; j++) acc[rt][dt][i2 + j] = mma_i8(p, vv[dt][j], acc[rt][dt][i2 + j]);
                        }
                };
                // a weight has a fourth limb from 0.498 on
                multiply(0, 3);
                if (__builtin_amdgcn_readfirstlane(int(l.top[buf][i]))) multiply(3, 4);
#pragma unroll
                for (int dt = 0; dt < 2; dt++)
#pragma unroll
                    for (int j = 0; j < 4; j++) vv[dt][j] = vn[dt][j];
            }
            if (sb + 1 < n_super) {
                load_numerators(e, sb + 1);
                park_weights(e, buf ^ 1);
            }
            __syncthreads();
        }
    }
    // at most 32768 keys: a sum of each worth is below 2^31, those of neighbouring worths together below 2^53
#pragma unroll
    for (int rt = 0; rt < 2; rt++)
#pragma unroll
        for (int dt = 0; dt < 2; dt++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const auto &s = acc[rt][dt];
                const double lo = __builtin_fma(__builtin_fma(double(s[2][i]), 0x1p8, double(s[1][i])), 0x1p8, double(s[0][i]));
                const double hi = __builtin_fma(__builtin_fma(__builtin_fma(double(s[6][i]), 0x1p8, double(s[5][i])), 0x1p8, double(s[4][i])), 0x1p8, double(s[3][i]));
                l.out[rt * 16 + 4 * g + i][wave * 32 + dt * 16 + c16] = float(__builtin_fma(hi, 0x1p24, lo) * 0x1p-48);
            }
}
// A tile of a head's positions from t0 on, in limbs (the queries' are in LDS) or in f64
template <uint32_t ROWS, bool LIMBS>
__device__ __forceinline__ void prompt_tile(const PromptArgs &a, PromptLds<ROWS> &l, uint32_t head, uint32_t kvh, uint32_t rank, uint32_t t0, float *s_row0) {
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = uint32_t(__builtin_amdgcn_readfirstlane(int(tid >> 6)));
    const uint32_t rows = a.n_tok - t0 < ROWS ? a.n_tok - t0 : ROWS;
    const uint32_t n_keys = a.step0 + t0 + rows;  // of the tile's last position
    // ---- 1
    const uint64_t tab_entry = kRmiExp2fTab[tid & 31];
    if constexpr (LIMBS)
        limb_scores(a, l, kvh, t0, rows, s_row0);
    else
        wide_scores<ROWS>(a, l, head, kvh, t0, rows, s_row0);
    if (tid < 32) l.exp_tab[tid] = tab_entry;
    __syncthreads();

    // ---- 2: numerators and their ordered sum.  A thread takes eight or sixteen keys of one position a turn; the sums are the
    // first wave's, or the third's of a workgroup that shares its compute unit with one whose first wave has them: the two
    // are on different SIMDs then
    {
        constexpr uint32_t kAcross = kThreads / ROWS * 4;  // keys that the threads of a position take at once
        const uint32_t r = tid / (kThreads / ROWS), k4 = tid % (kThreads / ROWS) * 4, last = a.step0 + t0 + (r < rows ? r : rows - 1);
        const bool sums = wave == (rank < a.half_tiles ? 0u : 2u) && lane < ROWS;
        const float max_val = fmaxf(fmaxf(l.row_max[0][r], l.row_max[1][r]), fmaxf(l.row_max[2][r], l.row_max[3][r]));
        float *src = s_row0 + size_t(r) * a.score_stride + k4;
        auto at = [&](uint32_t turn_i, uint32_t j) -> float4 & { return *reinterpret_cast<float4 *>(src + turn_i * kTurn + j * kAcross); };
        const uint32_t n_turns = (n_keys + kTurn - 1) / kTurn;
        float4 next[kTurn / kAcross];
#pragma unroll
        for (uint32_t j = 0; j < kTurn / kAcross; j++) next[j] = at(0, j);
        float acc = 0.0f;
        for (uint32_t turn_i = 0; turn_i <= n_turns; turn_i++) {
            if (turn_i < n_turns) {
                const uint32_t ahead = turn_i + 1 < n_turns ? turn_i + 1 : turn_i;
                const bool behind = (turn_i + 1) * kTurn > a.step0 + t0 + 1;  // keys that a position does not see among them
#pragma unroll
                for (uint32_t j = 0; j < kTurn / kAcross; j++) {
                    const float4 sc = next[j];
                    next[j] = at(ahead, j);
                    const float x[4] = {sc.x - max_val, sc.y - max_val, sc.z - max_val, sc.w - max_val};
                    float4 e;
                    if constexpr (!LIMBS)
                        e = {rmi_expf_tab(x[0], l.exp_tab), rmi_expf_tab(x[1], l.exp_tab), rmi_expf_tab(x[2], l.exp_tab), rmi_expf_tab(x[3], l.exp_tab)};
                    else
                        e = {rmi_expf_nonpositive(x[0], l.exp_tab), rmi_expf_nonpositive(x[1], l.exp_tab), rmi_expf_nonpositive(x[2], l.exp_tab), rmi_expf_nonpositive(x[3], l.exp_tab)};
                    if (behind) {
                        const uint32_t key = turn_i * kTurn + k4 + j * kAcross;
                        e.x = key <= last ? e.x : 0.0f;
                        e.y = key + 1 <= last ? e.y : 0.0f;
                        e.z = key + 2 <= last ? e.z : 0.0f;
                        e.w = key + 3 <= last ? e.w : 0.0f;
                    }
                    at(turn_i, j) = e;
                    *reinterpret_cast<float4 *>(&l.turn[turn_i & 1][r][k4 + j * kAcross]) = e;
                }
            }
            if (turn_i > 0 && sums) {  // the turn before: the reference adds the numerators one after the other in f32
                const float4 *p = reinterpret_cast<const float4 *>(l.turn[(turn_i - 1) & 1][lane]);
#pragma unroll
                for (uint32_t half = 0; half < 2; half++) {
                    float4 v[kTurn / 8];
#pragma unroll
                    for (uint32_t j = 0; j < kTurn / 8; j++) v[j] = p[half * (kTurn / 8) + j];
#pragma unroll
                    for (uint32_t j = 0; j < kTurn / 8; j++) {
                        acc += v[j].x;
                        acc += v[j].y;
                        acc += v[j].z;
                        acc += v[j].w;
                    }
                }
            }
            __syncthreads();
        }
        if (sums) l.row_sum[lane] = acc;
    }
    __syncthreads();

    // ---- 3
    if constexpr (LIMBS)
        limb_values(a, l, kvh, t0, rows, s_row0);
    else
        wide_values<ROWS>(a, l, kvh, t0, rows, s_row0);
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < ROWS / 8; k++) {  // four dimensions a thread: whole groups of eight lanes for the quantizer
        const uint32_t r = k * 8 + (tid >> 5), d4 = (tid & 31) * 4;
        float sc;
        const uint32_t packed = rmi_quantize_block8(*reinterpret_cast<const float4 *>(&l.out[r][d4]), a.rounding, &sc);
        if (r < rows) {
            const size_t first = (size_t(t0 + r) * a.n_head + head) * 128;
            reinterpret_cast<uint32_t *>(a.q8)[(first + d4) >> 2] = packed;
            if ((tid & 7) == 0) a.scales[(first + d4) >> 5] = sc;
        }
    }
}

// Which head and tile a launch's workgroup takes: key/value head fastest, so that with eight of them every workgroup that
// reads a head's keys is on one XCD
struct PromptPlace {
    uint32_t kvh, head, rank, tile;
};
__device__ __forceinline__ PromptPlace prompt_place(const PromptArgs &a, uint32_t i) {
    const uint32_t kvh = i % a.n_head_kv, hpk = a.n_head / a.n_head_kv, rank = i / a.n_head;
    return {kvh, kvh * hpk + (i / a.n_head_kv) % hpk, rank, a.first_tile + prompt_tile_of(rank, a.n_tiles, a.half_tiles)};
}
__global__ __launch_bounds__(kThreads, 2) void attn128_prompt_kernel(PromptArgs a) {
    __shared__ PromptLds<16> l;
    const PromptPlace p = prompt_place(a, blockIdx.x);
    prompt_tile<16, false>(a, l, p.head, p.kvh, p.rank, p.tile * 16, a.scratch + size_t(blockIdx.x) * 16 * a.score_stride);
}
// 32 positions a workgroup, in limbs where they hold.  In f64 those are a longer chain than sixteen, which tells where a
// compute unit has no other workgroup: there (gridDim.y = 2) such a tile is two workgroups' of sixteen, and the workgroups
// y = 1, whose tiles are in the other order, end at once otherwise.
__global__ __launch_bounds__(kThreads, 2) void attn128_prompt_limbs_kernel(PromptArgs a) {
    __shared__ union {
        PromptLds<kRows> whole;
        PromptLds<16> half;
    } l;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = uint32_t(__builtin_amdgcn_readfirstlane(int(tid >> 6)));
    const uint32_t c16 = lane & 15, g = lane >> 4, second = blockIdx.y;
    const uint32_t i = second ? (a.n_tiles - 1 - blockIdx.x / a.n_head) * a.n_head + blockIdx.x % a.n_head : blockIdx.x;
    const PromptPlace p = prompt_place(a, i);
    const uint32_t t0 = p.tile * kRows, rows = a.n_tok - t0 < kRows ? a.n_tok - t0 : kRows;
    const uint32_t n_blocks = (a.step0 + t0 + rows + 63) / 64;
    float *s_row0 = a.scratch + size_t(i) * kRows * a.score_stride;  // [position][key], rows of whole turns

    // Wave w: positions 16 (w / 2) .. + 15, half w % 2 of the dimensions, lane (c16, g) sixteen of them of position c16
    const uint32_t r = (wave >> 1) * 16 + c16, t = t0 + (r < rows ? r : rows - 1);
    const u32x4 *src = reinterpret_cast<const u32x4 *>(a.q16 + (size_t(t) * a.n_head + p.head) * 128 + (wave & 1) * 64 + g * 16);
    const u32x4 u[2] = {src[0], src[1]};
    bool wide = false;
    for (uint32_t b = tid; b < n_blocks; b += kThreads)
        wide |= (a.limbs.wide[p.kvh * a.limbs.blocks + b] | a.limbs.wide[(a.n_head_kv + p.kvh) * a.limbs.blocks + b]) != 0;
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int k = 0; k < 4; k++) wide |= !limbs_hold(u[j][k]);
    {
        _Float16 h[16];
#pragma unroll
        for (int j = 0; j < 16; j++) h[j] = __builtin_bit_cast(f16x8, u[j >> 3])[j & 7];
        u32x4 ql[4];
        limbs_of16(h, ql);
#pragma unroll
        for (int j = 0; j < 4; j++) l.whole.q[wave][j][lane] = ql[j];
    }
    wide = __syncthreads_or(wide);  // the same in both workgroups of a tile
    if (!wide) {
        if (second == 0) prompt_tile<kRows, true>(a, l.whole, p.head, p.kvh, p.rank, t0, s_row0);
    } else if (gridDim.y == 1) {
        prompt_tile<kRows, false>(a, l.whole, p.head, p.kvh, p.rank, t0, s_row0);
    } else if (second * 16 < rows) {
        prompt_tile<16, false>(a, l.half, p.head, p.kvh, p.rank, t0 + second * 16, s_row0 + size_t(second) * 16 * a.score_stride);
    }
}

// Whether a pass's keys and values are split into limbs: the splitting is a launch of 5 to 7 us that the products have to
// win back, and a head of values that limbs don't hold has it for nothing and its positions in f64.  So only where norms keep
// queries and keys small, and from a million products of a query and a key on.  us a layer, f64 | limbs, 16 heads: prompt of
// 128 99 | 103, 256 139 | 140, 384 184 | 182, 700 299 | 277, 1024 394 | 349; 2048 tokens in passes of 65 141 | 132, of 512 265 |
// 228, of 1024 476 | 380; 32 heads: prompt of 192 581 | 584, 256 691 | 690, 512 1215 | 1193, 1024 2428 | 2336.  Values that
// don't fit, 16 heads, in f64 from the start | found here: prompt of 384 196 | 204, 512 223 | 225 (216 and 245 with 32 positions a
// workgroup), 700 310 | 330, 1024 409 | 419, 2048 977 | 974.
bool limbs_pay(uint32_t n_head, uint32_t step0, uint32_t n_tok) { return uint64_t(n_head) * n_tok * (step0 + n_tok / 2) >= 1u << 20; }

}  // namespace

size_t rmi_attn_limbs_bytes(uint32_t n_head_kv, uint32_t capacity) { return size_t((capacity + 63) / 64) * n_head_kv * 2 * (kLimbBlock + 4); }
RmiAttnLimbs rmi_attn_limbs_at(void *base, uint32_t n_head_kv, uint32_t capacity) {
    if (!base) return RmiAttnLimbs{};
    const uint32_t blocks = (capacity + 63) / 64;
    const size_t plane = size_t(blocks) * n_head_kv * kLimbBlock;
    uint8_t *p = static_cast<uint8_t *>(base);
    return RmiAttnLimbs{p, p + plane, reinterpret_cast<uint32_t *>(p + 2 * plane), blocks};
}

bool rmi_attn_prompt_in_limbs(uint32_t n_head, uint32_t step0, uint32_t n_tok, const RmiAttnLimbs &limbs, bool limbs_hold) {
    return limbs.blocks && limbs_hold && step0 + n_tok <= kAttnLimbKeys && limbs_pay(n_head, step0, n_tok);
}
int rmi_launch_attn128_prompt(const uint16_t *q16, const uint16_t *k_cache, const uint16_t *v_cache, uint32_t step0, uint32_t n_tok,
                              uint32_t kv_stride, uint32_t n_head, uint32_t n_head_kv, float *scratch, size_t scratch_floats,
                              const RmiAttnLimbs &limbs, bool limbs_hold, int8_t *q8, float *scales, int rounding, hipStream_t st) {
    const uint32_t cus = uint32_t(rmi_device_cus()), stride = rmi_attn_prompt_score_stride(step0 + n_tok);
    const bool use_limbs = rmi_attn_prompt_in_limbs(n_head, step0, n_tok, limbs, limbs_hold);
    const uint32_t rows = use_limbs ? kRows : 16, tiles = (n_tok + rows - 1) / rows;
    const size_t tile_floats = size_t(n_head) * rows * stride;
    const uint32_t most = uint32_t(scratch_floats / tile_floats);  // tiles a launch has scratch for
    if (most == 0) return rmi_fail(RMI_HIP_E_INVALID, "%u keys exceed the scratch of a prompt pass", step0 + n_tok);
    if (use_limbs)
        hipLaunchKernelGGL(attn128_limbs_kernel, dim3((step0 + n_tok + 63) / 64, n_head_kv, 2), dim3(kThreads), 0, st, k_cache, v_cache, step0 + n_tok,
                           kv_stride, limbs);
    for (uint32_t t = 0; t < tiles; t += most) {
        const uint32_t n = tiles - t < most ? tiles - t : most;
        // workgroups that are all under way at once, two a compute unit: the second one's tiles in the other order
        const uint32_t half = n * n_head <= 2 * cus && n * n_head > cus ? (cus + n_head - 1) / n_head : n;
        const PromptArgs args{q16, k_cache, v_cache, step0, n_tok, kv_stride, n_head, n_head_kv, t, n, half, stride, scratch, q8, scales, rounding, limbs};
        if (use_limbs)
            hipLaunchKernelGGL(attn128_prompt_limbs_kernel, dim3(n * n_head, n * n_head <= cus ? 2 : 1), dim3(kThreads), 0, st, args);
        else
            hipLaunchKernelGGL(attn128_prompt_kernel, dim3(n * n_head), dim3(kThreads), 0, st, args);
    }
    RMI_HIP_CHECK(hipGetLastError());
    return RMI_HIP_OK;
}
