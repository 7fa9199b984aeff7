// Attention of a prompt pass over the F16 cache, head dimension 128 (src/models/qwen3.rs:876-933): many positions of a
// head at once, with the bits that attention128_quant_kernel gives each of them alone.
//
// The reference's rounding points are kept: f16 queries, keys and values; scores as f64 sums of exact products rounded
// to f32 and scaled; the softmax numerators by the libm's expf; their sum in f32, key after key; one f32 division a
// weight, rounded to f16; the weighted values as f64 sums of exact products.  The order of the two f64 sums is free (a
// product of two f16 has 22 bits, so sums over a few thousand of them are exact but for a rounding of about 2^-53), which
// lets both be matrix products: v_mfma_f64_16x16x4 with sixteen positions as its rows.
//
// A workgroup of four waves takes sixteen consecutive positions of one query head:
//   1  scores of sixteen keys a wave and turn into a row of scratch a position (at 2000 keys the rows of an XCD's workgroups,
//      8 MB, are twice its L2), and each position's maximum;
//   2  numerators, 64 keys of all sixteen positions a turn; lane r of the first wave adds position r's in order;
//   3  weights and p . v, sixteen keys a wave and turn; the waves' sums meet in LDS, then the quantizer.
// What bounds it: the matrix cores at f64 (64 clocks an instruction: 75 TFLOP/s), two of the four products of a
// position and key pair that a flash-style kernel would spend being saved by keeping the scores; the ordered sum is
// sixteen chains side by side on one wave, hidden behind the other workgroup of the compute unit.  Measured (16 heads, 512
// positions): 46 us over the first 512 keys, 178 us at 2000 keys, half of the f64 rate; the kernel before it, a workgroup
// a position and head on the vector ALU, took 31 us for 128 positions of the first 512 and went position by position from
// 1280 keys on (a prompt of 1999 tokens, 28 layers: 885 -> 47.5 ms, one of 512 and 32 answers: 37.4 -> 33.0 ms);
// it still does passes of up to 1024 positions times heads (pass_by_positions in decode_qwen3.hip).
#include "attn_prompt.h"

#include "device_math.h"
#include "device_quant.h"

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr uint32_t kThreads = 256, kRows = kAttnPromptRows, kTurn = 64;  // kTurn: keys of a turn of phase 2
constexpr uint32_t kTurnStride = kTurn + 4;                             // floats; four lanes' 16-byte reads on different banks

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

__global__ __launch_bounds__(kThreads, 2) void attn128_prompt_kernel(const uint16_t *__restrict__ q16, const uint16_t *__restrict__ k_cache,
                                                                     const uint16_t *__restrict__ v_cache, uint32_t step0, uint32_t n_tok,
                                                                     uint32_t kv_stride, uint32_t n_head, uint32_t n_head_kv,
                                                                     uint32_t first_tile, float *__restrict__ scratch, uint32_t score_stride,
                                                                     int8_t *__restrict__ q8, float *__restrict__ scales, int rounding) {
    __shared__ double part[3][kRows][128];  // phase 3; phase 2's turns lie in it
    __shared__ float row_max[4][kRows], row_sum[kRows];
    __shared__ uint64_t exp_tab[32];
    float (*turn)[kRows][kTurnStride] = reinterpret_cast<float (*)[kRows][kTurnStride]>(part);
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = uint32_t(__builtin_amdgcn_readfirstlane(int(tid >> 6)));
    const uint32_t c16 = lane & 15, g = lane >> 4;
    // key/value head fastest: with eight of them every workgroup that reads a head's cache rows is on one XCD
    const uint32_t kvh = blockIdx.x % n_head_kv, hpk = n_head / n_head_kv;
    const uint32_t head = kvh * hpk + (blockIdx.x / n_head_kv) % hpk;
    const uint32_t tile = first_tile + blockIdx.x / n_head;
    const uint32_t t0 = tile * kRows;                                        // first position of the tile, within the pass
    const uint32_t rows = n_tok - t0 < kRows ? n_tok - t0 : kRows;
    const uint32_t n_keys = step0 + t0 + rows;                               // of the tile's last position
    const uint32_t key_tiles = (n_keys + 15) / 16;
    float *s_row0 = scratch + size_t(blockIdx.x) * kRows * score_stride;     // [position][key], rows of whole turns
    const uint64_t tab_entry = kRmiExp2fTab[tid & 31];

    // ---- 1: scores.  Lane (c16, g) gives the matrix cores dimensions (4 c + g) * 8 .. + 7, c = 0..3, of position
    // (as A) or key (as B) c16: sixteen bytes a load, four lanes of a key 64 consecutive bytes
    f16x8 qh[4];
    {
        const uint32_t t = t0 + (c16 < rows ? c16 : rows - 1);
        const uint16_t *src = q16 + (size_t(t) * n_head + head) * 128 + g * 8;
#pragma unroll
        for (int c = 0; c < 4; c++) qh[c] = *reinterpret_cast<const f16x8 *>(src + c * 32);
    }
    const uint16_t *kbase = k_cache + size_t(kvh) * 128 + g * 8, *vbase = v_cache + size_t(kvh) * 128 + c16 * 8;
    auto load_keys = [&](f16x8 (&kk)[4], uint32_t kt) {  // (past the last position: that one again, masked below)
        const uint32_t key = kt * 16 + c16 < n_keys ? kt * 16 + c16 : n_keys - 1;
        const uint16_t *src = kbase + size_t(key) * kv_stride;
#pragma unroll
        for (int c = 0; c < 4; c++) kk[c] = *reinterpret_cast<const f16x8 *>(src + c * 32);
    };
    const float kq_scale = 1.0f / sqrtf(128.0f);  // two f32 roundings, as the reference computes it
    float my_max[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    f16x8 kk[4], kn[4];
    load_keys(kk, wave);
    for (uint32_t kt = wave; kt < key_tiles; kt += 4) {
        load_keys(kn, kt + 4);
        f64x4 s[2] = {{0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0}};
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int j = 0; j < 8; j++)
                s[j & 1] = __builtin_amdgcn_mfma_f64_16x16x4f64(half_f64(qh[c], j), half_f64(kk[c], j), s[j & 1], 0, 0, 0);
        const uint32_t key = kt * 16 + c16;
#pragma unroll
        for (int i = 0; i < 4; i++) {  // position 4 i + g of the tile, key c16
            const uint32_t r = 4 * i + g;
            const float sc = float(s[0][i] + s[1][i]) * kq_scale;
            if (key <= step0 + t0 + r) my_max[i] = fmaxf(my_max[i], sc);
            s_row0[size_t(r) * score_stride + key] = sc;
        }
#pragma unroll
        for (int c = 0; c < 4; c++) kk[c] = kn[c];
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        float m = my_max[i];
        m = fmaxf(m, dpp_f32<kDppQuadXor1>(m));
        m = fmaxf(m, dpp_f32<kDppQuadXor2>(m));
        m = fmaxf(m, dpp_f32<kDppRowHalfMirror>(m));
        m = fmaxf(m, dpp_f32<kDppRowMirror>(m));
        if (c16 == 0) row_max[wave][4 * i + g] = m;
    }
    if (tid < 32) exp_tab[tid] = tab_entry;
    __syncthreads();

    // ---- 2: numerators and their ordered sum.  A thread takes four keys of one position a turn
    const uint32_t n_turns = (n_keys + kTurn - 1) / kTurn;
    {
        const uint32_t r = tid >> 4, k4 = (tid & 15) * 4, last = step0 + t0 + r;
        const float max_val = fmaxf(fmaxf(row_max[0][r], row_max[1][r]), fmaxf(row_max[2][r], row_max[3][r]));
        float4 *src = reinterpret_cast<float4 *>(s_row0 + size_t(r) * score_stride) + (tid & 15);
        float4 next = src[0];
        float acc = 0.0f;
        for (uint32_t turn_i = 0; turn_i <= n_turns; turn_i++) {
            if (turn_i < n_turns) {
                const float4 sc = next;
                if (turn_i + 1 < n_turns) next = src[(turn_i + 1) * (kTurn / 4)];
                const uint32_t key = turn_i * kTurn + k4;
                float4 e;
                e.x = key <= last ? rmi_expf_tab(sc.x - max_val, exp_tab) : 0.0f;
                e.y = key + 1 <= last ? rmi_expf_tab(sc.y - max_val, exp_tab) : 0.0f;
                e.z = key + 2 <= last ? rmi_expf_tab(sc.z - max_val, exp_tab) : 0.0f;
                e.w = key + 3 <= last ? rmi_expf_tab(sc.w - max_val, exp_tab) : 0.0f;
                src[turn_i * (kTurn / 4)] = e;
                *reinterpret_cast<float4 *>(&turn[turn_i & 1][r][k4]) = e;
            }
            if (turn_i > 0 && tid < kRows) {  // the turn before: the reference adds the numerators one after the other in f32
                const float4 *p = reinterpret_cast<const float4 *>(turn[(turn_i - 1) & 1][tid]);
                float4 v[kTurn / 4];
#pragma unroll
                for (uint32_t j = 0; j < kTurn / 4; j++) v[j] = p[j];
#pragma unroll
                for (uint32_t j = 0; j < kTurn / 4; j++) {
                    acc += v[j].x;
                    acc += v[j].y;
                    acc += v[j].z;
                    acc += v[j].w;
                }
            }
            __syncthreads();
        }
        if (tid < kRows) row_sum[tid] = acc;
    }
    __syncthreads();

    // ---- 3: weights and values.  Lane (c16, g): weights of position c16 and keys 4 g .. 4 g + 3 of the sixteen (as A);
    // dimensions 8 c16 .. + 7 of the same keys (as B), so that product j's columns are the dimensions 8 c16 + j.  A key
    // behind a position has weight zero there, which hides its value as long as that is finite (0 x inf is NaN, which the
    // quantizer drops): of the few keys that some positions of the tile see and others do not, other values are taken out
    // and counted afterwards.
    f64x4 acc[8];
#pragma unroll
    for (int j = 0; j < 8; j++) acc[j] = f64x4{0.0, 0.0, 0.0, 0.0};
    {
        const float total = row_sum[c16];
        const uint32_t last = step0 + t0 + c16;
        const float4 *wsrc = reinterpret_cast<const float4 *>(s_row0 + size_t(c16) * score_stride) + g;
        auto load_values = [&](f16x8 (&vv)[4], float4 &e, uint32_t kt) {
            kt = kt < key_tiles ? kt : key_tiles - 1;
            e = wsrc[kt * 4];
#pragma unroll
            for (uint32_t i = 0; i < 4; i++) {
                const uint32_t key = kt * 16 + 4 * g + i < n_keys ? kt * 16 + 4 * g + i : n_keys - 1;
                vv[i] = *reinterpret_cast<const f16x8 *>(vbase + size_t(key) * kv_stride);
            }
        };
        auto weight = [&](float ev, uint32_t key) {
            const float w32 = total > 0.0f ? ev / total : ev;
            return key <= last ? double(h2f(rmi_f2h(w32))) : 0.0;
        };
        f16x8 vv[4], vn[4];
        float4 e, en;
        bool odd = false;
        load_values(vv, e, wave);
        for (uint32_t kt = wave; kt < key_tiles; kt += 4) {
            load_values(vn, en, kt + 4);
            const float ev[4] = {e.x, e.y, e.z, e.w};
            if (kt * 16 + 15 > step0 + t0) odd |= take_out_nonfinite(vv);
#pragma unroll
            for (uint32_t i = 0; i < 4; i++) {
                const double w = weight(ev[i], kt * 16 + 4 * g + i);
#pragma unroll
                for (int j = 0; j < 8; j++) acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(w, half_f64(vv[i], j), acc[j], 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < 4; i++) vv[i] = vn[i];
            e = en;
        }
        if (__any(odd))  // what was taken out, one position after the other, without the values behind it
            for (uint32_t kt = wave; kt < key_tiles; kt += 4) {
                if (kt * 16 + 15 <= step0 + t0) continue;
#pragma unroll 1
                for (uint32_t r = 0; r < rows; r++)
#pragma unroll 1
                    for (uint32_t i = 0; i < 4; i++) {
                        const uint32_t key = kt * 16 + 4 * g + i, there = key < n_keys ? key : n_keys - 1;
                        const double w = weight(s_row0[size_t(c16) * score_stride + key], key);
                        const f16x8 v = *reinterpret_cast<const f16x8 *>(vbase + size_t(there) * kv_stride);
#pragma unroll
                        for (int j = 0; j < 8; j++) {
                            const bool finite = fabsf(float(v[j])) <= 65504.0f;
                            const f64x4 o = __builtin_amdgcn_mfma_f64_16x16x4f64(w, finite || key > step0 + t0 + r ? 0.0 : half_f64(v, j), f64x4{0.0, 0.0, 0.0, 0.0}, 0, 0, 0);
#pragma unroll
                            for (uint32_t q = 0; q < 4; q++) acc[j][q] += 4 * q + g == r ? o[q] : 0.0;
                        }
                    }
            }
    }
    // lane (c16, g), register i: position 4 i + g, dimensions 8 c16 + j
    if (wave > 0) {
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 8; j++) part[wave - 1][4 * i + g][8 * c16 + j] = acc[j][i];
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 8; j++) part[0][4 * i + g][8 * c16 + j] = ((acc[j][i] + part[0][4 * i + g][8 * c16 + j]) + part[1][4 * i + g][8 * c16 + j]) + part[2][4 * i + g][8 * c16 + j];
    }
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < 2; k++) {  // four dimensions a thread: whole groups of eight lanes for the quantizer
        const uint32_t r = k * 8 + (tid >> 5), d4 = (tid & 31) * 4;
        const double *o = &part[0][r][d4];
        float sc;
        const uint32_t packed = rmi_quantize_block8(make_float4(float(o[0]), float(o[1]), float(o[2]), float(o[3])), rounding, &sc);
        if (r < rows) {
            const size_t first = (size_t(t0 + r) * n_head + head) * 128;
            reinterpret_cast<uint32_t *>(q8)[(first + d4) >> 2] = packed;
            if ((tid & 7) == 0) scales[(first + d4) >> 5] = sc;
        }
    }
}

}  // namespace

int rmi_launch_attn128_prompt(const uint16_t *q16, const uint16_t *k_cache, const uint16_t *v_cache, uint32_t step0, uint32_t n_tok,
                              uint32_t kv_stride, uint32_t n_head, uint32_t n_head_kv, float *scratch, size_t scratch_floats, int8_t *q8,
                              float *scales, int rounding, hipStream_t st) {
    const uint32_t tiles = (n_tok + kRows - 1) / kRows, stride = rmi_attn_prompt_score_stride(step0 + n_tok);
    const size_t tile_floats = size_t(n_head) * kRows * stride;
    const uint32_t most = uint32_t(scratch_floats / tile_floats);  // tiles a launch has scratch for
    if (most == 0) return rmi_fail(RMI_HIP_E_INVALID, "%u keys exceed the scratch of a prompt pass", step0 + n_tok);
    for (uint32_t t = 0; t < tiles; t += most) {
        const uint32_t n = tiles - t < most ? tiles - t : most;
        hipLaunchKernelGGL(attn128_prompt_kernel, dim3(n * n_head), dim3(kThreads), 0, st, q16, k_cache, v_cache, step0, n_tok, kv_stride, n_head,
                           n_head_kv, t, scratch, stride, q8, scales, rounding);
    }
    RMI_HIP_CHECK(hipGetLastError());
    return RMI_HIP_OK;
}
