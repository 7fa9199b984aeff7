// Products of several tokens on dense bf16 / f32 weights: the inputs (norms) in front of them, a tiled matrix-core
// GEMM with the layer's elementwise work in its epilogue (activations, gates, gated residual), and the embedding.
#include <type_traits>

#include "dense_launch.h"

namespace {

template <typename T, int NORM, bool ADD, int R>
__global__ __launch_bounds__(256) void input_kernel(RmiInput in, const uint32_t *__restrict__ rows, T *__restrict__ h, uint32_t k_pad,
                                                    uint32_t ld) {
    __shared__ float red[12];
    InputRow<NORM, ADD, R> r;
    const uint32_t row = rows ? rows[blockIdx.x] : blockIdx.x;
    r.load(in, row);
    r.finish(in, row, in.x_out != nullptr, red);
    if (h) r.store(in, row, h + size_t(blockIdx.x) * ld, k_pad);
}

template <typename T>
__global__ __launch_bounds__(256) void embed_kernel(RmiEmbed e, const uint32_t *__restrict__ tok, uint32_t pos0) {
    embed_row<T>(e, tok[blockIdx.x], pos0 + blockIdx.x, blockIdx.x);
}

template <typename T>
__global__ __launch_bounds__(256) void embed_token_kernel(RmiEmbed e, uint32_t token, uint32_t *tok, uint32_t pos) {
    if (threadIdx.x == 0) *tok = token;
    embed_row<T>(e, token, pos, 0);
}

// ------------------------------------------------------------------ GEMM
// Weights are the A operand: a lane ends with four consecutive rows of one token.  k goes in steps of 128 bytes a row
// through LDS; a row of a buffer is eight 16-byte pieces, piece p at slot p ^ (row & 7), so that the sixteen rows of a
// fragment spread over the banks.
constexpr uint32_t kStepBytes = 128;
constexpr uint32_t kSplitSteps = 4;  // of small tiles: steps of a round, the unit in which k is divided
constexpr uint32_t kMaxSplit = 16;
constexpr int kResidual = -1;  // the epilogue that adds to the residual stream; the others are RmiEpilogue's

// A wave's results, NN x NT tiles of sixteen rows x sixteen tokens: a lane has rows 4 g .. 4 g + 3 of one token of each.
// A finished column segment goes to the residual stream at once (each element is one thread's), so that no second set
// of accumulators is held.  row, tok: of the lane's first value.
template <int NN, int NT>
__device__ __forceinline__ void fold_segment(f32x4 (&acc)[NN][NT], const RmiColSeg &s, float *__restrict__ x, uint32_t width, uint32_t n_tokens,
                                             uint32_t row0, uint32_t tok0) {
    const bool quads = (width & 3) == 0;
#pragma unroll
    for (int j = 0; j < NT; j++) {
        const uint32_t tok = tok0 + j * 16;
#pragma unroll
        for (int i = 0; i < NN; i++) {
            const uint32_t row = row0 + i * 16;
            const size_t at = size_t(tok) * width + row;
            if (tok < n_tokens && row < width) {
                if (quads) {
                    f32x4 v = acc[i][j] * s.scale;
                    if (s.gate) v *= *reinterpret_cast<const f32x4 *>(s.gate + size_t(tok) * s.gate_ld + row);
                    *reinterpret_cast<f32x4 *>(x + at) += v;
                } else {
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        if (row + r < width) x[at + r] += acc[i][j][r] * s.scale * (s.gate ? s.gate[size_t(tok) * s.gate_ld + row + r] : 1.0f);
                }
            }
            acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
}

// first_row, tok0: of the wave's first tile and the lane's first token
template <typename T, int EPI, int NN, int NT>
__device__ __forceinline__ void store_rows(const f32x4 (&acc)[NN][NT], const RmiRowSegs &rs, uint32_t n_rows, uint32_t n_tokens, uint32_t first_row,
                                           uint32_t tok0, uint32_t g) {
#pragma unroll
    for (int i = 0; i < NN; i++) {
        const uint32_t tile_row = first_row + i * 16;  // a tile of sixteen rows lies in one segment
        if (tile_row >= n_rows) continue;
        const RmiRowSeg &s = rs.s[seg_of(rs, tile_row)];
        const uint32_t r0 = tile_row - s.row0 + g * 4;
        float bias[4], lower[4];
        if constexpr (EPI == kRowsActed || EPI == kRowsTimesTable) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
                bias[r] = s.bias && r0 + r < s.n ? s.bias[r0 + r] : 0.0f;
                lower[r] = s.lower && r0 + r < s.n ? s.lower[r0 + r] : 0.0f;
            }
        }
#pragma unroll
        for (int j = 0; j < NT; j++) {
            const uint32_t tok = tok0 + j * 16;
            if constexpr (EPI == kRowsPaired) {  // (gate, up) twice: two results
                if (tok >= n_tokens) continue;
                const f32x4 z = acc[i][j];
                const float v0 = fmaxf(z[0], 0.0f) * z[1], v1 = fmaxf(z[2], 0.0f) * z[3];
                const size_t at = size_t(tok) * s.ld + r0 / 2;
                if (sizeof(T) == 2 && s.out_elem && r0 + 2 < s.n && (s.ld & 1) == 0) {  // side by side: one store
                    reinterpret_cast<uint32_t *>(s.y)[at >> 1] = uint32_t(f32_to_bf16(v0)) | uint32_t(f32_to_bf16(v1)) << 16;
                    continue;
                }
#pragma unroll
                for (uint32_t r = 0; r < 2; r++) {
                    const float v = r ? v1 : v0;
                    if (r0 + 2 * r < s.n) {
                        if (s.out_elem)
                            static_cast<T *>(s.y)[at + r] = from_f32<T>(v);
                        else
                            static_cast<float *>(s.y)[at + r] = v;
                    }
                }
                continue;
            }
            f32x4 o = acc[i][j];
            if constexpr (EPI == kRowsActed || EPI == kRowsTimesTable) {
#pragma unroll
                for (int r = 0; r < 4; r++) o[r] = apply_act<T>(s.act, o[r], bias[r], lower[r]);
            }
            if (tok >= n_tokens) continue;
            if constexpr (EPI == kRowsTimesTable) {
                if (s.mul) {
                    const T *m = mul_row<T>(s, tok) + r0;
#pragma unroll
                    for (uint32_t r = 0; r < 4; r++)
                        if (r0 + r < s.n) o[r] *= to_f32(m[r]);
                }
            }
            const size_t at = size_t(tok) * s.ld + r0;
            if (r0 + 3 < s.n && (s.ld & 3) == 0) {
                if (s.out_elem)
                    store4(static_cast<T *>(s.y) + at, o);
                else
                    store4(static_cast<float *>(s.y) + at, o);
            } else {
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (r0 + r < s.n) {
                        if (s.out_elem)
                            static_cast<T *>(s.y)[at + r] = from_f32<T>(o[r]);
                        else
                            static_cast<float *>(s.y)[at + r] = o[r];
                    }
            }
        }
    }
}

// The same results by whole lines: sixteen tokens at a time through LDS of the wave's own, from where a lane takes four
// consecutive rows of one token and its neighbours the rows beside them.  From the registers a token's stores are 64 bytes (32
// in bf16) of a line here and the rest of it in later instructions, and the code is written out for every tile of sixteen by
// sixteen: with the activations more than the instruction cache holds, a miss a line in every wave.  Of 256 x 256 tiles in bf16
// (activated, 39168 x 4096, 2048 tokens) 213 of 690 us were this epilogue; 146 of them are left (268 MB of f32 and bf16 results, and the
// activations).  Segments are whole groups
// of sixteen rows, so a lane's rows are one's; where the wave's rows are of several it goes through them one by one.
// tile: 16 (WN + 4) floats.
template <typename T, int EPI, int WN, int NN, int NT>
__device__ __forceinline__ void store_lines(const f32x4 (&acc)[NN][NT], const RmiRowSegs &rs, uint32_t n_tokens, uint32_t first_row, uint32_t tok_first,
                                            float *tile) {
    constexpr uint32_t kLanes = WN / 4, kAtOnce = 64 / kLanes, kLd = WN + 4;  // lanes of a token, tokens of an instruction
    constexpr bool kActs = EPI == kRowsActed || EPI == kRowsTimesTable;
    const uint32_t lane = threadIdx.x & 63, fr = lane & 15, g = lane >> 4, r = lane % kLanes * 4;
    for (uint32_t si = uint32_t(__builtin_amdgcn_readfirstlane(int(seg_of(rs, first_row)))); si < rs.n_segs; si++) {
        const RmiRowSeg &s = rs.s[si];
        if (s.row0 >= first_row + WN) break;
        const uint32_t r0 = first_row + r - s.row0;  // (rows in front of the segment are far behind its end)
        const bool whole = r0 < s.n && s.n - r0 >= 4 && (s.ld & 3) == 0;
        f32x4 bias = {0.f, 0.f, 0.f, 0.f}, lower = bias;
        if constexpr (kActs) {
#pragma unroll
            for (uint32_t e = 0; e < 4; e++) {
                if (s.bias && r0 < s.n) bias[e] = s.bias[r0 + e < s.n ? r0 + e : s.n - 1];
                if (s.lower && r0 < s.n) lower[e] = s.lower[r0 + e < s.n ? r0 + e : s.n - 1];
            }
        }
        auto sixteen = [&](int j, auto act_c) {
#pragma unroll 2
            for (uint32_t t = lane / kLanes; t < 16; t += kAtOnce) {
                f32x4 o = *reinterpret_cast<const f32x4 *>(tile + t * kLd + r);
                const uint32_t tok = tok_first + j * 16 + t;
                if (tok >= n_tokens || r0 >= s.n) break;
                if constexpr (EPI == kRowsPaired) {  // (gate, up) twice: two results
                    const float v0 = fmaxf(o[0], 0.0f) * o[1], v1 = fmaxf(o[2], 0.0f) * o[3];
                    const size_t at = size_t(tok) * s.ld + r0 / 2;
                    if (sizeof(T) == 2 && s.out_elem && r0 + 2 < s.n && (s.ld & 1) == 0) {  // side by side: one store
                        reinterpret_cast<uint32_t *>(s.y)[at >> 1] = uint32_t(f32_to_bf16(v0)) | uint32_t(f32_to_bf16(v1)) << 16;
                    } else {
#pragma unroll
                        for (uint32_t e = 0; e < 2; e++)
                            if (r0 + 2 * e < s.n) {
                                if (s.out_elem)
                                    static_cast<T *>(s.y)[at + e] = from_f32<T>(e ? v1 : v0);
                                else
                                    static_cast<float *>(s.y)[at + e] = e ? v1 : v0;
                            }
                    }
                } else {
                    if constexpr (kActs) {
#pragma unroll
                        for (int e = 0; e < 4; e++) o[e] = apply_act<T>(decltype(act_c)::value, o[e], bias[e], lower[e]);
                    }
                    if constexpr (EPI == kRowsTimesTable) {
                        if (s.mul) {
                            const T *m = mul_row<T>(s, tok) + r0;
#pragma unroll
                            for (uint32_t e = 0; e < 4; e++)
                                if (r0 + e < s.n) o[e] *= to_f32(m[e]);
                        }
                    }
                    const size_t at = size_t(tok) * s.ld + r0;
                    if (whole) {
                        if (s.out_elem)
                            store4(static_cast<T *>(s.y) + at, o);
                        else
                            store4(static_cast<float *>(s.y) + at, o);
                    } else {
#pragma unroll
                        for (uint32_t e = 0; e < 4; e++)
                            if (r0 + e < s.n) {
                                if (s.out_elem)
                                    static_cast<T *>(s.y)[at + e] = from_f32<T>(o[e]);
                                else
                                    static_cast<float *>(s.y)[at + e] = o[e];
                            }
                    }
                }
            }
        };
#pragma unroll
        for (int j = 0; j < NT; j++) {
#pragma unroll
            for (int i = 0; i < NN; i++) *reinterpret_cast<f32x4 *>(tile + fr * kLd + i * 16 + g * 4) = acc[i][j];
            rmi_wave_lds_fence();
            switch (kActs ? s.act : uint16_t(kActNone)) {
            case kActSigmoid: sixteen(j, std::integral_constant<uint32_t, kActSigmoid>{}); break;
            case kActSilu: sixteen(j, std::integral_constant<uint32_t, kActSilu>{}); break;
            case kActGeluTanh: sixteen(j, std::integral_constant<uint32_t, kActGeluTanh>{}); break;
            case kActForgetGate: sixteen(j, std::integral_constant<uint32_t, kActForgetGate>{}); break;
            default: sixteen(j, std::integral_constant<uint32_t, kActNone>{});
            }
            rmi_wave_lds_fence();
        }
    }
}

// The same for a product that joins x: what is there and the gates are asked for together, in front of the tiles' way through
// LDS.
template <int WN, int NT>
struct ResidualLines {
    static constexpr uint32_t kLanes = WN / 4, kAtOnce = 64 / kLanes, kLd = WN + 4, kTimes = 16 / kAtOnce;
    f32x4 v[NT][kTimes], gate[NT][kTimes];

    static __device__ __forceinline__ uint32_t row_of(uint32_t first_row) { return first_row + (threadIdx.x & 63) % kLanes * 4; }
    static __device__ __forceinline__ uint32_t tok_of(uint32_t tok_first, int j, uint32_t k) { return tok_first + j * 16 + k * kAtOnce + (threadIdx.x & 63) / kLanes; }
    __device__ __forceinline__ void load(const RmiColSeg &s, const float *x, uint32_t width, uint32_t n_tokens, uint32_t first_row, uint32_t tok_first) {
        const uint32_t row = row_of(first_row) < width ? row_of(first_row) : width - 4;
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (uint32_t k = 0; k < kTimes; k++) {
                const uint32_t t = tok_of(tok_first, j, k), tok = t < n_tokens ? t : n_tokens - 1;
                v[j][k] = *reinterpret_cast<const f32x4 *>(x + size_t(tok) * width + row);
                gate[j][k] = f32x4{1.f, 1.f, 1.f, 1.f};
                if (s.gate) gate[j][k] = *reinterpret_cast<const f32x4 *>(s.gate + size_t(tok) * s.gate_ld + row);
            }
    }
    template <int NN>
    __device__ __forceinline__ void add(const f32x4 (&acc)[NN][NT], const RmiColSeg &s, float *x, uint32_t width, uint32_t n_tokens, uint32_t first_row,
                                        uint32_t tok_first, float *tile) {
        const uint32_t lane = threadIdx.x & 63, fr = lane & 15, g = lane >> 4, row = row_of(first_row);
#pragma unroll
        for (int j = 0; j < NT; j++) {
#pragma unroll
            for (int i = 0; i < NN; i++) *reinterpret_cast<f32x4 *>(tile + fr * kLd + i * 16 + g * 4) = acc[i][j];
            rmi_wave_lds_fence();
#pragma unroll
            for (uint32_t k = 0; k < kTimes; k++) {
                const f32x4 o = *reinterpret_cast<const f32x4 *>(tile + (k * kAtOnce + lane / kLanes) * kLd + lane % kLanes * 4);
                const uint32_t tok = tok_of(tok_first, j, k);
                if (tok < n_tokens && row < width) *reinterpret_cast<f32x4 *>(x + size_t(tok) * width + row) = v[j][k] + o * s.scale * gate[j][k];
            }
            rmi_wave_lds_fence();
        }
    }
};

// What a column segment adds to the residual stream, onto z, and the accumulators at zero again.
template <int NN, int NT>
__device__ __forceinline__ void gather_segment(f32x4 (&acc)[NN][NT], f32x4 (&z)[NN][NT], const RmiColSeg &s, uint32_t width, uint32_t n_tokens, uint32_t row0,
                                               uint32_t tok0) {
    const bool quads = (width & 3) == 0;
#pragma unroll
    for (int j = 0; j < NT; j++) {
        const uint32_t tok = tok0 + j * 16;
#pragma unroll
        for (int i = 0; i < NN; i++) {
            const uint32_t row = row0 + i * 16;
            f32x4 gate = {1.f, 1.f, 1.f, 1.f};
            if (s.gate && tok < n_tokens && row < width) {
                const float *at = s.gate + size_t(tok) * s.gate_ld + row;
                if (quads) {
                    gate = *reinterpret_cast<const f32x4 *>(at);
                } else {
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        if (row + r < width) gate[r] = at[r];
                }
            }
            z[i][j] += acc[i][j] * s.scale * gate;
            acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
}
template <int NN, int NT>
__device__ __forceinline__ void join_stream(const f32x4 (&z)[NN][NT], float *__restrict__ x, uint32_t width, uint32_t n_tokens, uint32_t row0, uint32_t tok0) {
    const bool quads = (width & 3) == 0;
#pragma unroll
    for (int j = 0; j < NT; j++) {
        const uint32_t tok = tok0 + j * 16;
#pragma unroll
        for (int i = 0; i < NN; i++) {
            const uint32_t row = row0 + i * 16;
            if (tok >= n_tokens || row >= width) continue;
            const size_t at = size_t(tok) * width + row;
            if (quads) {
                *reinterpret_cast<f32x4 *>(x + at) += z[i][j];
            } else {
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (row + r < width) x[at + r] += z[i][j][r];
            }
        }
    }
}

// A tile's k over `parts` workgroups.  Each leaves its sums (past the caches, as the parts' workgroups sit on any XCD); the one that
// counts last adds all of them, in the parts' order, and goes on to the epilogue.  Nobody waits for another.
struct DenseParts {
    uint32_t parts, tiles;
    uint32_t *counts;  // one a tile, zero before and after
    float *sums;       // [tile][part][values of a thread, by twos][thread]
};
template <int NN, int NT>
__device__ __forceinline__ bool parts_meet(f32x4 (&v)[NN][NT], const DenseParts &dp, uint32_t tile, uint32_t part, uint32_t *last) {
    constexpr uint32_t kPairs = NN * NT * 2, kPart = kPairs * 256;
    uint64_t *all = reinterpret_cast<uint64_t *>(dp.sums) + size_t(tile) * dp.parts * kPart + threadIdx.x, *mine = all + size_t(part) * kPart;
#pragma unroll
    for (uint32_t k = 0; k < kPairs; k++) {
        const f32x4 &q = v[k / 2 / NT][k / 2 % NT];
        const uint64_t pair = uint64_t(__float_as_uint(q[k % 2 * 2])) | uint64_t(__float_as_uint(q[k % 2 * 2 + 1])) << 32;
        __hip_atomic_store(mine + k * 256, pair, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the stores are out before the count says so)
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t n = __hip_atomic_fetch_add(dp.counts + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *last = n == dp.parts - 1;
        if (n == dp.parts - 1) __hip_atomic_store(dp.counts + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next launch
    }
    __syncthreads();
    if (!*last) return false;
#pragma unroll
    for (int i = 0; i < NN; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) v[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto add = [&](auto at_a_time, uint32_t p0) {  // parts whose loads are under way together
        constexpr uint32_t N = at_a_time.value;
        uint64_t pair[N][kPairs];
#pragma unroll
        for (uint32_t p = 0; p < N; p++)
#pragma unroll
            for (uint32_t k = 0; k < kPairs; k++)
                pair[p][k] = __hip_atomic_load(all + size_t(p0 + p) * kPart + k * 256, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (uint32_t p = 0; p < N; p++)
#pragma unroll
            for (uint32_t k = 0; k < kPairs; k++) {
                f32x4 &q = v[k / 2 / NT][k / 2 % NT];
                q[k % 2 * 2] += __uint_as_float(uint32_t(pair[p][k]));
                q[k % 2 * 2 + 1] += __uint_as_float(uint32_t(pair[p][k] >> 32));
            }
    };
    uint32_t p = 0;
    for (; p + 4 <= dp.parts; p += 4) add(std::integral_constant<uint32_t, 4>(), p);
    for (; p < dp.parts; p++) add(std::integral_constant<uint32_t, 1>(), p);
    return true;
}

// Four waves; the pieces of the next PD steps are on their way to registers while one is multiplied.  Small tiles, for
// products that would leave compute units idle otherwise, have two LDS buffers; 128 x 128 keeps one (NB = 1), so that three
// workgroups share a compute unit: one round where wider tiles would start a second one for a few workgroups.
template <typename T, int BN, int BT, int WN, int WT, int PD, int NB, int WPS, int EPI, bool SPLIT = false>
__global__ __launch_bounds__(256, WPS) void dense_gemm_kernel(const T *__restrict__ w, const T *__restrict__ a, uint32_t n_rows,
                                                              uint32_t k_pad, uint32_t ld, uint32_t n_tokens, uint32_t grid_n, uint32_t grid_t, uint32_t xcd_split,
                                                         RmiRowSegs rs, RmiColSegs cs, float *__restrict__ x, uint32_t width, DenseParts dp) {
    constexpr bool RESIDUAL = EPI == kResidual;
    static_assert((BN / WN) * (BT / WT) == 4, "four waves");
    static_assert(kDenseKAlign * sizeof(T) % (kStepBytes * PD) == 0, "whole rounds of the register slots");
    constexpr int NN = WN / 16, NT = WT / 16;
    constexpr int PW = BN * 8 / 256, PA = (BT * 8 + 255) / 256;  // pieces a thread loads per step
    __shared__ u32x4 lds[NB][(BN + BT) * 8];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = uint32_t(__builtin_amdgcn_readfirstlane(int(tid >> 6)));
    const uint32_t part = SPLIT ? blockIdx.x / dp.tiles : 0, tile = blockIdx.x - part * dp.tiles;
    uint32_t n_tile, t_tile;
    rmi_gemm_tile_of(tile, grid_n, grid_t, 1u, xcd_split, n_tile, t_tile);
    const uint32_t row0 = n_tile * BN, tok0 = t_tile * BT;
    const uint32_t wn = (wave % (BN / WN)) * WN, wt = (wave / (BN / WN)) * WT;
    const size_t stride = size_t(ld) * sizeof(T);

    const uint8_t *wsrc[PW], *asrc[PA];
    uint32_t wdst[PW], adst[PA];
#pragma unroll
    for (int i = 0; i < PW; i++) {
        const uint32_t e = tid + i * 256, r = e >> 3, p = e & 7;
        const uint32_t row = row0 + r < n_rows ? row0 + r : n_rows - 1;  // rows past the end are read again and not stored
        wsrc[i] = reinterpret_cast<const uint8_t *>(w) + row * stride + p * 16;
        wdst[i] = r * 8 + (p ^ (r & 7));
    }
#pragma unroll
    for (int i = 0; i < PA; i++) {
        const uint32_t e = tid + i * 256, r = (e >> 3) % BT, p = e & 7;  // (fewer pieces than threads: some load twice)
        const uint32_t tok = tok0 + r < n_tokens ? tok0 + r : n_tokens - 1;
        asrc[i] = reinterpret_cast<const uint8_t *>(a) + tok * stride + p * 16;
        adst[i] = BN * 8 + r * 8 + (p ^ (r & 7));
    }
    f32x4 acc[NN][NT];
#pragma unroll
    for (int i = 0; i < NN; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    constexpr uint32_t kStepElems = kStepBytes / sizeof(T);
    const uint32_t n_steps = k_pad / kStepElems, rounds = n_steps / PD;
    const uint32_t first = SPLIT ? part * rounds / dp.parts * PD : 0, end = SPLIT ? (part + 1) * rounds / dp.parts * PD : n_steps;
    u32x4 rw[PD][PW], ra[PD][PA];
    auto load = [&](int slot, uint32_t step) {
        // always issued (past the end the last step again): the waits count loads, and a skipped one would make every
        // wait a wait for all
        step = step < end ? step : end - 1;
#pragma unroll
        for (int i = 0; i < PW; i++) rw[slot][i] = *reinterpret_cast<const u32x4 *>(wsrc[i] + size_t(step) * kStepBytes);
#pragma unroll
        for (int i = 0; i < PA; i++) ra[slot][i] = *reinterpret_cast<const u32x4 *>(asrc[i] + size_t(step) * kStepBytes);
    };
    auto park = [&](int slot, uint32_t buf) {
#pragma unroll
        for (int i = 0; i < PW; i++) lds[buf][wdst[i]] = rw[slot][i];
#pragma unroll
        for (int i = 0; i < PA; i++) lds[buf][adst[i]] = ra[slot][i];
    };
    const uint32_t fr = lane & 15, g = lane >> 4;
#pragma unroll
    for (int j = 0; j < PD; j++) {
        load(j, first + j);
        asm volatile("" ::: "memory");  // in this order, and here: the waits in the loop count on it
    }
    park(0, 0);
    load(0, first + PD);
    asm volatile("" ::: "memory");
    __syncthreads();
    uint32_t step = first;
    constexpr bool kGather = SPLIT && RESIDUAL;
    f32x4 z[NN][NT];  // what a part's segments add
    if constexpr (kGather) {
#pragma unroll
        for (int i = 0; i < NN; i++)
#pragma unroll
            for (int j = 0; j < NT; j++) z[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    for (uint32_t seg = 0; seg < (RESIDUAL ? cs.n_segs : 1u); seg++) {
        // segments end at multiples of kDenseKAlign, whole rounds of the register slots
        const uint32_t k_end = RESIDUAL ? cs.s[seg].k_end / kStepElems : n_steps, seg_end = SPLIT && end < k_end ? end : k_end;
        if (SPLIT && seg_end <= step) continue;
        for (; step < seg_end; step += PD) {
#pragma unroll
            for (int j = 0; j < PD; j++) {  // register slots by compile-time index
                const uint32_t buf = (step + j) & (NB - 1);
#pragma unroll
                for (int c = 0; c < 2; c++) {
                    u32x4 fw[NN], fa[NT];
#pragma unroll
                    for (int i = 0; i < NN; i++) {
                        const uint32_t r = wn + i * 16 + fr;
                        fw[i] = lds[buf][r * 8 + ((c * 4 + g) ^ (r & 7))];
                    }
#pragma unroll
                    for (int i = 0; i < NT; i++) {
                        const uint32_t r = wt + i * 16 + fr;
                        fa[i] = lds[buf][BN * 8 + r * 8 + ((c * 4 + g) ^ (r & 7))];
                    }
#pragma unroll
                    for (int i = 0; i < NN; i++)
#pragma unroll
                        for (int i2 = 0; i2 < NT; i2++) acc[i][i2] = mma16<T>(fw[i], fa[i2], acc[i][i2]);
                }
                if (NB == 1) __syncthreads();
                park((j + 1) % PD, buf ^ (NB - 1));  // (behind the last step: that step again, read by nobody)
                load((j + 1) % PD, step + j + 1 + PD);
                __syncthreads();
            }
        }
        if constexpr (kGather)
            gather_segment<NN, NT>(acc, z, cs.s[seg], width, n_tokens, row0 + wn + g * 4, tok0 + wt + fr);
        else if constexpr (RESIDUAL)
            fold_segment<NN, NT>(acc, cs.s[seg], x, width, n_tokens, row0 + wn + g * 4, tok0 + wt + fr);
    }

    if constexpr (SPLIT) {
        __shared__ uint32_t last;
        bool here;
        if constexpr (RESIDUAL)
            here = parts_meet<NN, NT>(z, dp, tile, part, &last);
        else
            here = parts_meet<NN, NT>(acc, dp, tile, part, &last);
        if (!here) return;
    }
    if constexpr (kGather) join_stream<NN, NT>(z, x, width, n_tokens, row0 + wn + g * 4, tok0 + wt + fr);
    if constexpr (!RESIDUAL) store_rows<T, EPI, NN, NT>(acc, rs, n_rows, n_tokens, row0 + wn, tok0 + wt + fr, g);
}

// s_waitcnt's operand: at most vm loads outstanding, and no LDS instruction
constexpr int rmi_waitcnt(int vm) { return (vm & 15) | (vm >> 4) << 14 | 7 << 4; }

// The same product with wider tiles and eight waves, so that a piece read from LDS feeds more products and the operands
// cross the L2 less often.  Steps go from memory straight into LDS (the swizzle is on the source side: a lane fetches the
// piece that belongs at its slot) through NB buffers, one barrier a step: behind it the next step's first half is read while
// the second half of this one is multiplied, and the buffer that everybody has read takes the step NB on.  The wait in front
// of the barrier counts the loads in flight, so that those of NB - 2 steps stay under way.
// What bounds it: the matrix cores at the clock that they have under full load, and the way from L2.  Of the 327 us of 128 x 256
// tiles (4096 x 20480, 2048 tokens, three column segments and so three launches) the products and barriers alone are 263 (1300
// TFLOP/s, what a large library product reaches); 256 x 256 tiles (39168 x 4096) run their loop in 474 us, 1386 TFLOP/s, in front of 146 us of results; 64 x 128
// tiles ask 96 bytes a clock and compute unit of L2, and take as long as that does.
template <typename T, int BN, int BT, int WN, int WT, int NB, int WPS, int EPI>
__global__ __launch_bounds__(64 * (BN / WN) * (BT / WT), WPS) void dense_gemm_wide_kernel(const T *__restrict__ w, const T *__restrict__ a, uint32_t n_rows, uint32_t k_pad,
                                                                 uint32_t ld, uint32_t n_tokens, uint32_t grid_n, uint32_t grid_t, uint32_t xcd_split,
                                                                 RmiRowSegs rs, RmiColSegs cs, float *__restrict__ x, uint32_t width) {
    constexpr bool RESIDUAL = EPI == kResidual;
    constexpr int NN = WN / 16, NT = WT / 16, WAVES = (BN / WN) * (BT / WT);
    constexpr int FW = BN / (8 * WAVES), FA = BT / (8 * WAVES);  // kilobytes a wave fetches of either operand per step: eight rows each
    __shared__ u32x4 buf0[(BN + BT) * 8], buf1[(BN + BT) * 8], buf2[NB == 3 ? (BN + BT) * 8 : 1];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = uint32_t(__builtin_amdgcn_readfirstlane(int(tid >> 6)));
    uint32_t n_tile, t_tile;
    rmi_gemm_tile_of(blockIdx.x, grid_n, grid_t, 1u, xcd_split, n_tile, t_tile);
    const uint32_t row0 = n_tile * BN, tok0 = t_tile * BT;
    const uint32_t wn = (wave % (BN / WN)) * WN, wt = (wave / (BN / WN)) * WT;
    const uint32_t stride = ld * uint32_t(sizeof(T));

    typedef const uint8_t __attribute__((address_space(1))) *gptr_u8;
    typedef __attribute__((address_space(3))) void *lptr;
    const gptr_u8 w_base = as_global<gptr_u8>(reinterpret_cast<const uint8_t *>(w) + size_t(row0) * stride);
    const gptr_u8 a_base = as_global<gptr_u8>(reinterpret_cast<const uint8_t *>(a) + size_t(tok0) * stride);
    uint32_t w_off[FW], a_off[FA];
    const uint32_t piece = ((lane & 7) ^ (lane >> 3)) * 16;  // of row lane >> 3 of eight, at slot lane & 7
#pragma unroll
    for (int i = 0; i < FW; i++) {
        const uint32_t r = (i * WAVES + wave) * 8 + (lane >> 3);
        w_off[i] = (row0 + r < n_rows ? r : n_rows - 1 - row0) * stride + piece;  // rows past the end are read again and not stored
    }
#pragma unroll
    for (int i = 0; i < FA; i++) {
        const uint32_t r = (i * WAVES + wave) * 8 + (lane >> 3);
        a_off[i] = (tok0 + r < n_tokens ? r : n_tokens - 1 - tok0) * stride + piece;
    }
    constexpr uint32_t kStepElems = kStepBytes / sizeof(T);
    const uint32_t first = RESIDUAL ? cs.k_begin / kStepElems : 0, n_steps = (RESIDUAL ? cs.s[0].k_end : k_pad) / kStepElems;
    auto fetch = [&](u32x4 *buf, uint32_t step) {
        const uint32_t at = (step < n_steps ? step : n_steps - 1) * kStepBytes;  // (behind the last step: that one again, read by nobody)
#pragma unroll
        for (int i = 0; i < FW; i++)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(w_base + (w_off[i] + at)), (lptr)(buf + (i * WAVES + wave) * 64), 16, 0, 0);
#pragma unroll
        for (int i = 0; i < FA; i++)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(a_base + (a_off[i] + at)), (lptr)(buf + BN * 8 + (i * WAVES + wave) * 64), 16, 0, 0);
    };
    const uint32_t fr = lane & 15, g = lane >> 4;
    f32x4 acc[NN][NT];
#pragma unroll
    for (int i = 0; i < NN; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    u32x4 fw[2][NN], fa[2][NT];
    auto read = [&](const u32x4 *buf, int c) {
        const uint32_t slot = (c * 4 + g) ^ (fr & 7);
#pragma unroll
        for (int i = 0; i < NN; i++) fw[c][i] = buf[(wn + i * 16 + fr) * 8 + slot];
#pragma unroll
        for (int j = 0; j < NT; j++) fa[c][j] = buf[BN * 8 + (wt + j * 16 + fr) * 8 + slot];
    };
    auto multiply = [&](int c) {
#pragma unroll
        for (int i = 0; i < NN; i++)
#pragma unroll
            for (int j = 0; j < NT; j++) acc[i][j] = mma16<T>(fw[c][i], fa[c][j], acc[i][j]);
    };
    static_assert(NB == 2 || NB == 3, "two or three buffers");
    // The order of what stands between two of these: one of the LDS reads (and of the loads) behind every product or two.  Left
    // to itself the compiler puts the reads behind the products, right in front of the wait for them (256 x 256, activated 39168 x
    // 4096, 2048 tokens: 720 -> 690 us).
    auto spread = [&](int loads) {
        constexpr int kReads = NN + NT, kProducts = NN * NT * int(sizeof(T) == 2 ? 1 : 4);
        constexpr int kEach = kProducts / (2 * kReads) > 0 ? kProducts / (2 * kReads) : 1;
#pragma unroll
        for (int i = 0; i < kReads; i++) {
#pragma unroll
            for (int n = 0; n < kEach; n++) __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if (i < loads) {
                __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, kProducts, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto step_of = [&](u32x4 *cur, u32x4 *next, uint32_t step) {
        read(cur, 1);
        multiply(0);
        spread(0);
        // this step is in everybody's registers, the next one in LDS; the loads of the one after it stay in flight
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(rmi_waitcnt((NB - 2) * (FW + FA)));
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        read(next, 0);
        fetch(cur, step + NB);
        multiply(1);
        spread(FW + FA);
    };
    fetch(buf0, first);
    fetch(buf1, first + 1);
    if constexpr (NB == 3) fetch(buf2, first + 2);
    __builtin_amdgcn_s_waitcnt(rmi_waitcnt((NB - 1) * (FW + FA)));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read(buf0, 0);
    // Whole turns of the buffers in a loop that has no other way out: with one, the compiler takes it that a buffer may be read
    // right behind its fetch, and waits for every load in flight once a turn (128 x 256, residual 4096 x 20480, 2048 tokens: 355 us with that, the
    // three segments in the loop and the results joining x from the registers; 327 without, in three launches).
    uint32_t step = first;
    auto buffer = [&](int i) { return i % NB == 0 ? buf0 : i % NB == 1 ? buf1 : buf2; };
    for (; step + NB <= n_steps; step += NB) {
#pragma unroll
        for (int i = 0; i < NB; i++) step_of(buffer(i), buffer(i + 1), step + i);
    }
    if (step < n_steps) step_of(buffer(0), buffer(1), step);
    if (NB == 3 && step + 1 < n_steps) step_of(buffer(1), buffer(2), step + 1);

    if (RESIDUAL && (width & 3)) {
        fold_segment<NN, NT>(acc, cs.s[0], x, width, n_tokens, row0 + wn + g * 4, tok0 + wt + fr);
        return;
    }
    __builtin_amdgcn_s_waitcnt(rmi_waitcnt(0));  // the steps behind the end are in LDS, and everybody has read the last one
    ResidualLines<WN, NT> there;
    if constexpr (RESIDUAL) there.load(cs.s[0], x, width, n_tokens, row0 + wn, tok0 + wt);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    constexpr uint32_t kTile = 16 * (WN + 4) / 4;  // in pieces; half of the waves' in either buffer
    static_assert(WAVES / 2 * kTile <= (BN + BT) * 8, "the waves' tiles fit the buffers");
    float *tile = reinterpret_cast<float *>((wave < WAVES / 2 ? buf0 : buf1) + wave % (WAVES / 2) * kTile);
    if constexpr (RESIDUAL)
        there.template add<NN>(acc, cs.s[0], x, width, n_tokens, row0 + wn, tok0 + wt, tile);
    else
        store_lines<T, EPI, WN, NN, NT>(acc, rs, n_tokens, row0 + wn, tok0 + wt, tile);
}

// Which tile a product takes: the least of estimates, in microseconds, that were fitted to every tile's time on 51 weights
// (64..39968 rows of 256..20480 columns; plain, activated, paired, table and residual ones) with 17..2048 tokens, each launch
// with a weight from HBM as in a model.  `fit` tiles run side by side on a compute unit and make a round.  A step of k takes
// `round` in a whole round; the tiles left over take `first`, and `more` and `whole` for what is beyond one a compute unit, by
// its share and by the whole tile.  An epilogue is not overlapped where a compute unit holds one workgroup, and adds to or
// activates a whole tile: so much a tile, which decides between wide tiles at 1024 columns.
// bf16 is bound by LDS reads and the traffic between L2 and the compute units, so wider tiles are cheaper an element as long
// as there are enough of them; f32 is bound by the matrix cores and every tile costs its area.  Over 597 products of bf16 and
// as many of f32 the choice costs 0.7 % and 0.03 % over the best tile of each (four waves alone: 6 and 5 %).  E.g. in bf16, us
// by 64 x 64 | 64 x 128 | 128 x 128 with four waves | with eight | 128 x 256 | 256 x 256:
//   activated 12304 x 1024, 2048 tokens    138 |  129 | 103 | 104 | 121 | 120     768 tokens    54 |  53 |  47 |  50 |  67 |  61
//   activated 39968 x 4096, 2048 tokens   1504 | 1169 | 797 | 846 | 760 | 687     512 tokens   320 | 280 | 210 | 231 | 233 | 264
//   residual 4096 x 12288, 2048 tokens     375 |  303 | 246 | 239 | 193 | 341     512 tokens   102 | 104 | 150 | 170 | 195 | 357
// All of that with results that left the wide tiles from the registers.  By lines they are faster (the first four rows with SiLU and
// results in bf16 now: 128 | 96 | 97 | 79 | 78 | 71 and 45 | 37 | 42 | 38 | 41 | 35, 1481 | 1080 | 770 | 741 | 599 | 528 and
// 315 | 252 | 202 | 227 | 181 | 207), which the estimates don't know: over 264 products of eleven weights the choice costs 5 % over
// the best tile, at most 40 %, nearly always by being narrower than that.
enum DenseTile { kTile64x16, kTile64x32, kTile64x64, kTile64x128, kTile128x128w4, kTile128x128, kTile128x256, kTile256x256 };
struct TileCost {
    DenseTile tile;
    uint32_t rows, tokens, waves, fit;
    float fixed, round, first, more, whole, out, activated, residual;
};
// 64 x 16 is what up to sixteen tokens take; its estimates only say over how many workgroups k goes
constexpr TileCost kTile16Bf16 = {kTile64x16, 64, 16, 4, 4, 4.0f, 0.66f, 0.165f, 0.07f, 0.1f, 0.2f, 0, 0};
constexpr TileCost kTile16F32 = {kTile64x16, 64, 16, 4, 4, 4.2f, 0.72f, 0.25f, 0.05f, 0.12f, 0.3f, 0, 0};
constexpr TileCost kCostsBf16[] = {
    {kTile64x32, 64, 32, 4, 4, 4.04f, 0.728f, 0.174f, 0.078f, 0.113f, 0.347f, 0, 0},
    {kTile64x64, 64, 64, 4, 4, 3.86f, 0.845f, 0.302f, 0.0412f, 0.154f, 1.08f, 1.81f, 0.973f},
    {kTile64x128, 64, 128, 8, 2, 3.78f, 0.809f, 0.525f, 0.123f, 0.184f, 0.789f, 1.14f, 0},
    {kTile128x128w4, 128, 128, 4, 3, 4.09f, 1.6f, 0.884f, 0, 0.308f, 2.44f, 4.23f, 0},
    {kTile128x128, 128, 128, 8, 2, 7.06f, 1.1f, 0.844f, 0.268f, 0, 0, 6.78f, 0},
    {kTile128x256, 128, 256, 8, 1, 7.53f, 0.947f, 0.882f, 0, 0, 4.05f, 12.6f, 0},
    {kTile256x256, 256, 256, 8, 1, 23.8f, 1.83f, 1.27f, 0, 0, 0, 24.5f, 0}};
constexpr TileCost kCostsF32[] = {
    {kTile64x32, 64, 32, 4, 4, 4.23f, 1.12f, 0.322f, 0.0836f, 0.187f, 0.438f, 0.803f, 0.103f},
    {kTile64x64, 64, 64, 4, 4, 4.36f, 1.96f, 0.588f, 0.0653f, 0.408f, 0.986f, 1.14f, 2.62f},
    {kTile64x128, 64, 128, 8, 2, 3.56f, 1.78f, 0.959f, 0, 0.845f, 2.04f, 2.0f, 6.56f},
    {kTile128x128, 128, 128, 8, 2, 6.12f, 3.54f, 1.81f, 0.04f, 1.67f, 2.36f, 5.63f, 16.2f}};

// k over several workgroups a tile (where the caller has memory for it): a workgroup takes its share of the steps, and the parts' sums cost a
// hand-over and a way out and back.  bf16 stays within a workgroup a compute unit, beyond which L2 bounds it; f32 is divided also where the
// tiles are a round and a bit, as the matrix cores bound it and the bit costs a whole one.  Three in a hundred at least are to be gained.
// us by the tile without parts | so: bf16 residual 1024 x 6144, 9 tokens 19.4 | 9.1, 40 tokens 19.6 | 9.5, 128 tokens 21.5 | 10.8, 300 tokens
// 20.2 | 18.2; 4096 x 12288, 64 tokens 45 | 29; f32 residual 2048 x 6144, 300 tokens 110 | 75, 1024 x 3072, 60 tokens 34 | 12; rows
// 128 x 2048, 300 tokens in f32 23.5 | 9.5.  Not divided: bf16 2048 x 12288, 512 tokens, 54 whole, 57 by two; f32 6144 x 2048, 300 tokens, 68, 76.
struct DenseChoice {
    const TileCost *tile;
    uint32_t parts;
};
DenseChoice dense_tile_of(bool bf16, int epilogue, uint32_t n_rows, uint32_t n_tokens, uint32_t n_steps, bool may_split) {
    const uint32_t cus = rmi_device_cus() > 0 ? uint32_t(rmi_device_cus()) : 1;
    DenseChoice best{nullptr, 1};
    double least = 0;
    auto consider = [&](const TileCost &c) {
        if (epilogue == kResidual && c.tile == kTile256x256) return;  // (2 % the better at the widest at most, and registers spilled, by the older way out)
        const uint64_t tiles = uint64_t((n_rows + c.rows - 1) / c.rows) * ((n_tokens + c.tokens - 1) / c.tokens);
        const uint32_t rounds = n_steps / kSplitSteps;
        for (uint32_t parts = 1; parts <= kMaxSplit; parts++) {
            const uint64_t groups = tiles * parts, sums = groups * c.rows * c.tokens;
            if (parts > 1 && (!may_split || c.tokens > 64 || parts > rounds || tiles > kDenseCounters || sums > kDenseSums || (bf16 && groups > cus))) break;
            const uint64_t full = groups / (c.fit * cus), left = groups % (c.fit * cus);
            double step = double(full) * c.round;
            if (left) step += c.first + c.whole * double((left - 1) / cus) + (left > cus ? c.more * (double(left) / cus - 1.0) : 0.0);
            const double end = c.out + (epilogue == kResidual ? c.residual : epilogue == kRowsActed || epilogue == kRowsTimesTable ? c.activated : 0.0f);
            double us = c.fixed + (parts == 1 ? n_steps : (rounds + parts - 1) / parts * kSplitSteps) * step + double(tiles) / cus * end;
            if (parts > 1) us = (us + 2.0 + double(sums) * 8 / 4.5e6) * 1.03;
            if (!best.tile || us < least) least = us, best = DenseChoice{&c, parts};
        }
    };
    if (n_tokens <= kTile16Bf16.tokens)
        consider(bf16 ? kTile16Bf16 : kTile16F32);
    else if (bf16)
        for (const TileCost &c : kCostsBf16) consider(c);
    else
        for (const TileCost &c : kCostsF32) consider(c);
    return best;
}

template <typename T, int EPI>
int launch_gemm(const RmiDense &w, const void *a, const RmiRowSegs &rs, const RmiColSegs &cs, float *x, uint32_t width,
                uint32_t n_tokens, const RmiDenseWork *work, hipStream_t st) {
    const uint32_t n_rows = EPI == kResidual ? width : w.n_rows;
    const DenseChoice choice = dense_tile_of(sizeof(T) == 2, EPI, n_rows, n_tokens, uint32_t(w.k_pad * sizeof(T) / kStepBytes), work != nullptr);
    const TileCost &tile = *choice.tile;
    const uint32_t gn = (n_rows + tile.rows - 1) / tile.rows, gt = (n_tokens + tile.tokens - 1) / tile.tokens;
    const uint32_t split = rmi_gemm_xcd_split(gn, gt, double(n_rows) * w.k_pad, double(n_tokens) * w.k_pad);
    auto launch = [&](auto kernel, uint32_t blocks, const RmiColSegs &c, auto... more) {
        hipLaunchKernelGGL(kernel, dim3(blocks), dim3(64 * tile.waves), 0, st, static_cast<const T *>(w.data), static_cast<const T *>(a), n_rows,
                           w.k_pad, w.ld, n_tokens, gn, gt, split, rs, c, x, width, more...);
    };
    auto go = [&](auto whole, auto in_parts) {
        const DenseParts dp{choice.parts, gn * gt, work ? work->counts : nullptr, work ? work->sums : nullptr};
        if (choice.parts > 1)
            launch(in_parts, gn * gt * choice.parts, cs, dp);
        else
            launch(whole, gn * gt, cs, dp);
    };
    auto go_wide = [&](auto kernel) {  // a launch for every column segment
        if constexpr (EPI != kResidual) {
            launch(kernel, gn * gt, cs);
        } else {
            for (uint32_t i = 0; i < cs.n_segs; i++) {
                RmiColSegs one{};
                one.s[0] = cs.s[i];
                one.n_segs = 1;
                one.k_begin = i ? cs.s[i - 1].k_end : 0;
                launch(kernel, gn * gt, one);
            }
        }
    };
    switch (tile.tile) {
    case kTile64x16: go(dense_gemm_kernel<T, 64, 16, 16, 16, kSplitSteps, 2, 4, EPI>, dense_gemm_kernel<T, 64, 16, 16, 16, kSplitSteps, 2, 4, EPI, true>); break;
    case kTile64x32: go(dense_gemm_kernel<T, 64, 32, 32, 16, kSplitSteps, 2, 4, EPI>, dense_gemm_kernel<T, 64, 32, 32, 16, kSplitSteps, 2, 4, EPI, true>); break;
    case kTile64x64: go(dense_gemm_kernel<T, 64, 64, 32, 32, kSplitSteps, 2, 4, EPI>, dense_gemm_kernel<T, 64, 64, 32, 32, kSplitSteps, 2, 4, EPI, true>); break;
    case kTile64x128: go_wide(dense_gemm_wide_kernel<T, 64, 128, 32, 32, 3, 2, EPI>); break;
    case kTile128x128: go_wide(dense_gemm_wide_kernel<T, 128, 128, 64, 32, 2, 4, EPI>); break;
    default:
        if constexpr (sizeof(T) == 2) {
            if (tile.tile == kTile128x128w4) launch(dense_gemm_kernel<T, 128, 128, 64, 64, 1, 1, 3, EPI>, gn * gt, cs, DenseParts{});
            if (tile.tile == kTile128x256) go_wide(dense_gemm_wide_kernel<T, 128, 256, 64, 64, 3, 2, EPI>);
            if constexpr (EPI != kResidual)
                if (tile.tile == kTile256x256) go_wide(dense_gemm_wide_kernel<T, 256, 256, 128, 64, 2, 2, EPI>);
        }
    }
    RMI_HIP_CHECK(hipGetLastError());
    return RMI_HIP_OK;
}

}  // namespace

uint32_t rmi_dense_tile(uint32_t elem_bytes, int epilogue, uint32_t n_rows, uint32_t k_pad, uint32_t n_tokens) {
    const TileCost &t = *dense_tile_of(elem_bytes == 2, epilogue, n_rows, n_tokens, k_pad * elem_bytes / kStepBytes, false).tile;
    return t.rows << 16 | t.tokens << 4 | t.waves;
}

uint32_t rmi_dense_parts(uint32_t elem_bytes, int epilogue, uint32_t n_rows, uint32_t k_pad, uint32_t n_tokens) {
    const DenseChoice c = dense_tile_of(elem_bytes == 2, epilogue, n_rows, n_tokens, k_pad * elem_bytes / kStepBytes, true);
    return c.parts << 16 | c.tile->tokens << 4 | c.tile->waves;
}

int rmi_dense_input(uint32_t elem_bytes, const RmiInput &in, const uint32_t *rows, void *h, uint32_t n_tokens, uint32_t k_pad,
                    hipStream_t st) {
    if (n_tokens == 0) return RMI_HIP_OK;
    int rc = rmi_check_input(in, k_pad, h == nullptr);
    if (rc != RMI_HIP_OK) return rc;
    auto go = [&](auto type) {
        using T = decltype(type);
        return rmi_input_dispatch(in, [&](auto norm, auto add, auto r) {
            hipLaunchKernelGGL((input_kernel<T, norm.value, add.value, r.value>), dim3(n_tokens), dim3(256), 0, st, in, rows, static_cast<T *>(h),
                               k_pad, rmi_dense_ld(k_pad, sizeof(T)));
            return RMI_HIP_OK;
        });
    };
    rc = elem_bytes == 2 ? go(rmi_bf16()) : go(float());
    RMI_HIP_CHECK(hipGetLastError());
    return rc;
}

int rmi_dense_embed(uint32_t elem_bytes, const RmiEmbed &e, const uint32_t *tok, uint32_t pos0, uint32_t n_tokens, hipStream_t st) {
    if (n_tokens == 0) return RMI_HIP_OK;
    if (elem_bytes == 2)
        hipLaunchKernelGGL(embed_kernel<rmi_bf16>, dim3(n_tokens), dim3(256), 0, st, e, tok, pos0);
    else
        hipLaunchKernelGGL(embed_kernel<float>, dim3(n_tokens), dim3(256), 0, st, e, tok, pos0);
    RMI_HIP_CHECK(hipGetLastError());
    return RMI_HIP_OK;
}

int rmi_dense_embed_token(uint32_t elem_bytes, const RmiEmbed &e, uint32_t token, uint32_t *tok, uint32_t pos, hipStream_t st) {
    if (elem_bytes == 2)
        hipLaunchKernelGGL(embed_token_kernel<rmi_bf16>, dim3(1), dim3(256), 0, st, e, token, tok, pos);
    else
        hipLaunchKernelGGL(embed_token_kernel<float>, dim3(1), dim3(256), 0, st, e, token, tok, pos);
    RMI_HIP_CHECK(hipGetLastError());
    return RMI_HIP_OK;
}

int rmi_dense_gemm(uint32_t elem_bytes, const RmiDense &w, const void *a, const RmiRowSegs &segs, uint32_t n_tokens, const RmiDenseWork &work, hipStream_t st) {
    if (n_tokens == 0 || w.n_rows == 0) return RMI_HIP_OK;
    const int rc = rmi_check_row_segs(elem_bytes, w, segs);
    if (rc != RMI_HIP_OK) return rc;
    auto go = [&](auto type) {
        using T = decltype(type);
        switch (rmi_epilogue_of(segs)) {
            case kRowsActed: return launch_gemm<T, kRowsActed>(w, a, segs, RmiColSegs{}, nullptr, 0, n_tokens, work.counts ? &work : nullptr, st);
            case kRowsPaired: return launch_gemm<T, kRowsPaired>(w, a, segs, RmiColSegs{}, nullptr, 0, n_tokens, work.counts ? &work : nullptr, st);
            case kRowsTimesTable: return launch_gemm<T, kRowsTimesTable>(w, a, segs, RmiColSegs{}, nullptr, 0, n_tokens, work.counts ? &work : nullptr, st);
            default: return launch_gemm<T, kRowsPlain>(w, a, segs, RmiColSegs{}, nullptr, 0, n_tokens, work.counts ? &work : nullptr, st);
        }
    };
    return elem_bytes == 2 ? go(rmi_bf16()) : go(float());
}

int rmi_dense_gemm_residual(uint32_t elem_bytes, const RmiDense &w, const void *a, const RmiColSegs &segs, float *x, uint32_t width,
                            uint32_t n_tokens, const RmiDenseWork &work, hipStream_t st) {
    if (n_tokens == 0) return RMI_HIP_OK;
    const int rc = rmi_check_col_segs(elem_bytes, w, segs, width);
    if (rc != RMI_HIP_OK) return rc;
    return elem_bytes == 2 ? launch_gemm<rmi_bf16, kResidual>(w, a, RmiRowSegs{}, segs, x, width, n_tokens, work.counts ? &work : nullptr, st)
                           : launch_gemm<float, kResidual>(w, a, RmiRowSegs{}, segs, x, width, n_tokens, work.counts ? &work : nullptr, st);
}
