// Generated tokens of a Qwen3 session by one launch: a workgroup a compute unit, each with a role, that hand the vectors of a
// layer to one another through HBM's caches, layer after layer and token after token.
//
// A token by launches is 144 dependent ones.  Each takes 2.4 us before its first instruction has run and the last one's results
// can be read, another 0.8 to read them, and its weights are asked for only then; 0.70 ms a token of width 1024 and 28 layers,
// of which 0.1 is what HBM needs for the weights.  Here a boundary is one exchange (1.0 to 1.5 us from the last workgroup's words
// stored to the last one's read, with 64 to 256 workgroups that read 256 to 1024 words), and the weights of a workgroup's next
// product are in its registers before the vector arrives: they are loaded right behind the product before.
//
// Exchange: a word of 64 bits is 32 bits of a vector and the tag of (token, layer) that it belongs to, stored and loaded whole
// by relaxed atomics of agent scope; a reader asks until all its words have the tag.  No fence and no counter is needed:
// everything that crosses workgroups inside a launch does so in such words, except the cache rows of a position, which are
// stored through to memory and waited for ahead of the words that the next token depends on, and which no workgroup has read
// before.  A buffer is written again only by workgroups that have waited for words which depend on every reader of it:
//   x    residual -> norm     all norm workgroups' q|k|v words reach attention, whose words every residual workgroup awaits
//   qkv  norm -> attention    the next x depends on all of attention's words
//   att  attention -> residual, xm residual -> norm, h norm -> residual, top all -> residual: likewise one stage on
// Every wait is bounded: a wave that has asked `spins` times marks the launch as failed, which ends the others' waits too, and the
// session generates again by single launches.  The launch is a cooperative one: every workgroup has a place, whoever starts first.
//
// us a token, 28 layers and a vocabulary of 151936, by launches | walked: behind 100 keys 590 | 425, 700: 761 | 520, 1250: 932 | 685.
// What a layer takes, us behind 100 | 544 | 1200 keys: 13.8 | 16.9 | 21.9, of that five exchanges 6.0 | 6.1 | 6.0 (a word alone takes
// 0.4 to one's own XCD, 0.6 to another, and the last of 64 to 128 workgroups counts), two norms and quantizers 1.0, the four
// products and what follows them 3.7, attention 3.0 | 6.1 | 11.2: scores 0.8 | 1.8 | 2.9, their largest (from 352 keys on with a
// sixth exchange) 0.6 | 1.0 | 1.2, exp and the f32 sum in key order 0.7 | 2.2 | 4.2, weighted values 0.9 | 1.1 | 3.0.
//
// A workgroup's words go out before any of its waves asks for the next weights (the barriers in front of those loads): stores
// of a late wave queue behind the other waves' loads, and everybody waits for that wave's words.  Without the barriers, and with
// arrays in LDS that 16-byte reads found unaligned, the three were 460, 540 and 714.
//
// Roles.  attention: four workgroups a head, as in attention128_quant_kernel<true, 4>.  residual: the o and down products, two
// tiles of eight rows a workgroup and four waves a tile, the rows' residual stream in registers.  norm: rms_norm, quantizer and
// the q|k|v or gate|up products behind it.  All: the vocabulary projection.  Arithmetic, rounding points and the order of every
// f32 sum are those of the single launches (decode_qwen3.hip, gemv_q8_0.hip).
#include "walk_qwen3.h"

#include <cmath>

#include "device_attn128.h"
#include "device_math.h"
#include "device_octet.h"
#include "device_quant.h"
#include "device_run_ring.h"
#include "device_sample.h"
#include "device_walk.h"

namespace {

constexpr uint32_t kWalkThreads = 512;

// where the vectors of the exchange lie, in words.  Quantized ones by blocks of 32 values: eight words of four quants, the scale.
struct WalkWords {
    uint32_t x, qkv, att, xm, h, top, n;
    uint32_t scores;  // behind both copies of the others: a head's are its own workgroups' matter
};
__host__ __device__ inline WalkWords walk_words(uint32_t n_embd, uint32_t n_head, uint32_t n_head_kv, uint32_t n_ff, uint32_t n_wg) {
    WalkWords w;
    uint32_t at = 0;
    auto take = [&](uint32_t n) {
        const uint32_t a = at;
        at += (n + 15) / 16 * 16;
        return a;
    };
    w.x = take(n_embd);
    w.qkv = take((n_head + 2 * n_head_kv) * 128);
    w.att = take(n_head * 4 * 9);
    w.xm = take(n_embd);
    w.h = take(n_ff / 32 * 9);
    w.top = take(n_wg * 4);
    w.n = at;
    w.scores = 2 * at;
    return w;
}

// A quantized block of 32, held as rmi_quantize_block32 leaves it in a wave's two halves: a copy from each.
__device__ __forceinline__ void block_store(gptr_word at, uint32_t copy, uint32_t q, float scale, uint32_t tag) {
    const uint32_t lane = threadIdx.x & 63, e = lane & 31;
    if ((e & 3) == 0 || e == 1) word_store(at + (lane >> 5) * copy + (e == 1 ? 8 : e >> 2), e == 1 ? __float_as_uint(scale) : q, tag);
}
struct WalkLds {  // of every role
    double red[8];
    float gu[64];
    Top top[64];
    Top all_top[8];  // by wave, of all workgroups: not in `top`, which wave 0 may still be reading when another wave has its words
    uint32_t bad;
    alignas(16) uint16_t new16[3][128];  // (read by pieces of 16 bytes)
    uint64_t exp_tab[32];
    float max8[8];
};

// The norm's weights of this thread's four elements (of threads without any, the first four: an unconditional load)
template <int NE>
struct NormWeights {
    float4 w;
    __device__ __forceinline__ void load(const float *from) {
        const u32x4 v = as_global<gptr_u4>(from)[threadIdx.x < NE * 64 ? threadIdx.x : 0];
        w = make_float4(__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z), __uint_as_float(v.w));
    }
};
// rms_norm of the vector in `words` times its weights, quantized into the staged order of the octets (NE of them, then the
// scales).  All waves wait for words and square them; four elements a thread, half of the waves do the rest: with two elements in
// every thread each SIMD has the long chain (square root, three divisions) twice, 1.0 us in the place of 0.75.
template <int NE>
__device__ __forceinline__ bool stage_norm(gptr_word words, uint32_t tag, const NormWeights<NE> &wv, const RmiWalkArgs &a, uint4 *lds, WalkLds &sm) {
    constexpr int W = NE * 256 / int(kWalkThreads);
    const uint32_t tid = threadIdx.x;
    float *xs = reinterpret_cast<float *>(lds + NE * 18);
    gptr_word at[W];
    uint32_t v[W];
#pragma unroll
    for (int j = 0; j < W; j++) at[j] = words + j * kWalkThreads + tid;
    if (!words_wait<W>(at, tag, v, WalkBound{a.failed, a.spins})) sm.bad = 1;
    double part = 0.0;
#pragma unroll
    for (int j = 0; j < W; j++) {
        const float f = __uint_as_float(v[j]), s = f * f;
        xs[j * kWalkThreads + tid] = f;
        part += double(s);
    }
    part = wave_sum_f64(part);
    if ((tid & 63) == 0) sm.red[tid >> 6] = part;
    __syncthreads();
    if (sm.bad) return false;
    if (tid < NE * 64) {
        const float4 x = reinterpret_cast<const float4 *>(xs)[tid];
        const double total = ((sm.red[0] + sm.red[1]) + (sm.red[2] + sm.red[3])) + ((sm.red[4] + sm.red[5]) + (sm.red[6] + sm.red[7]));
        const float mean_sq = float(total / double(NE * 256));
        const float scale = 1.0f / sqrtf(mean_sq + a.eps);
        float4 o;
        o.x = (x.x * scale) * wv.w.x;
        o.y = (x.y * scale) * wv.w.y;
        o.z = (x.z * scale) * wv.w.z;
        o.w = (x.w * scale) * wv.w.w;
        float sc;
        const uint32_t q = rmi_quantize_block8(o, a.rounding, &sc);
        const uint32_t b = tid >> 3;  // block of this float4; tid & 7 = its dword inside the block
        uint32_t *dq = reinterpret_cast<uint32_t *>(lds);
        dq[(b >> 2) * 32 + (tid & 7) * 4 + (b & 3)] = q;
        if ((tid & 7) == 0) reinterpret_cast<float *>(dq + NE * 64)[b] = sc;
    }
    __syncthreads();
    return true;
}

// A quantized vector of n_oct octets out of its words into the staged order.
template <int MAXW>
__device__ __forceinline__ bool stage_quants(gptr_word words, uint32_t tag, uint32_t n_oct, const RmiWalkArgs &a, uint4 *lds, WalkLds &sm) {
    const uint32_t tid = threadIdx.x, n = n_oct * 72;
    gptr_word at[MAXW];
    uint32_t v[MAXW];
#pragma unroll
    for (int j = 0; j < MAXW; j++) {
        const uint32_t w = j * kWalkThreads + tid;
        at[j] = words + (w < n ? w : n - 1);
    }
    if (!words_wait<MAXW>(at, tag, v, WalkBound{a.failed, a.spins})) sm.bad = 1;
    uint32_t *dq = reinterpret_cast<uint32_t *>(lds);
#pragma unroll
    for (int j = 0; j < MAXW; j++) {
        const uint32_t w = j * kWalkThreads + tid, b = w / 9, l = w - b * 9;
        if (w < n) {
            const uint32_t dst = l < 8 ? (b >> 2) * 32 + l * 4 + (b & 3) : n_oct * 64 + b;
            dq[dst] = v[j];
        }
    }
    __syncthreads();
    return !sm.bad;
}

// Every workgroup: the vocabulary projection of the norm of x, the workgroup's largest logits to `top`.
template <int NE>
__device__ __forceinline__ bool walk_head(const RmiWalkArgs &a, const WalkWords &at, gptr_word words, gptr_word mine, uint32_t tag, bool keep, uint4 *lds,
                                          WalkLds &sm) {
    const uint32_t tid = threadIdx.x, lane = tid & 63, r = lane >> 3, L = lane & 7;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t n_tiles = (a.vocab + 7) / 8, n_waves = gridDim.x * 8, w_idx = blockIdx.x * 8 + wave;
    const uint32_t k0 = uint32_t(uint64_t(n_tiles) * w_idx / n_waves), k1 = uint32_t(uint64_t(n_tiles) * (w_idx + 1) / n_waves);
    const uint32_t n_units = (k1 - k0) * NE;
    struct Cursor {
        gptr_u4 sc_unit, q_unit;
        uint32_t o, r, lane;
        __device__ __forceinline__ void load(OctetRegs &g) const {
            g.sc = sc_unit[r];
            g.qa = __builtin_nontemporal_load(q_unit + lane);
            g.qb = __builtin_nontemporal_load(q_unit + 64 + lane);
        }
        __device__ __forceinline__ void step() {
            sc_unit += 8;
            q_unit += 128;
            if (++o == NE) {  // over this tile's quants / the next tile's scales
                o = 0;
                sc_unit += NE * 128;
                q_unit += NE * 8;
            }
        }
    } cur;
    gptr_u4 tile = as_global<gptr_u4>(a.head + size_t(n_units ? k0 : 0) * NE * kOctetBytes);
    cur = Cursor{tile, tile + NE * 8, 0, r, lane};
    RmiRing<OctetRegs> ring;
    rmi_ring_fill(ring, n_units, cur);
    NormWeights<NE> wv;
    wv.load(a.output_norm);
    if (!stage_norm<NE>(mine + at.x, tag, wv, a, lds, sm)) return false;
    Top t{-INFINITY, -INFINITY, 0xffffffffu, 1u};
    float acc[1] = {0.0f};
    uint32_t o = 0, k = k0;
    auto consume = [&](const OctetRegs &g) {
        octet_fma_one(acc[0], g, lds, NE, o, L);
        if (++o == NE) {
            const float y = hsum8_lanes(acc[0]);
            acc[0] = 0.0f;
            o = 0;
            const uint32_t row = k * 8 + r;
            if (row < a.vocab) {
                if (keep && L == 0) as_global<gptr_f32_w>(a.logits)[row] = y;
                if (!(fabsf(y) <= 3.4028234663852886e38f)) t.finite = 0;  // NaN or inf
                if (y > t.best) {
                    t.second = t.best;
                    t.best = y;
                    t.id = row;
                } else if (y > t.second) {
                    t.second = y;
                }
            }
            k++;
        }
    };
    rmi_ring_walk(ring, n_units, cur, consume);
    if (L == 0) sm.top[wave * 8 + r] = t;
    __syncthreads();
    if (tid < 64) {
        Top m = sm.top[tid];
#pragma unroll
        for (int s = 32; s > 0; s >>= 1) {
            const Top other{__shfl_xor(m.best, s), __shfl_xor(m.second, s), uint32_t(__shfl_xor(int(m.id), s)), uint32_t(__shfl_xor(int(m.finite), s))};
            m = top_merge(m, other);
        }
        if (tid < 8)
            word_store(words + (tid >> 2) * at.n + at.top + blockIdx.x * 4 + (tid & 3),
                       (tid & 3) == 0 ? __float_as_uint(m.best) : (tid & 3) == 1 ? __float_as_uint(m.second) : (tid & 3) == 2 ? m.id : m.finite, tag);
    }
    return true;
}

// ---- attention: workgroup `idx` of 4 n_head; key/value head fastest (attention128_quant_kernel has the layout's reasons).
// Eight lanes a key, lane8 takes the 16-byte pieces lane8 and 8 + lane8 of its 256 bytes.  The first three rounds of 64 keys are
// turned into f64 before this position's query is there: a product is one f64 fma then (exact terms, any order of them gives the
// same sum but for a last bit in 2^26), in the place of product, conversion and addition.
// From kWalkShareKeys keys on a head's four workgroups take a quarter of its keys' scores each and hand them to one another, 1.3 us
// for the exchange: us a layer without | with, 132 keys 15.9 | 16.3, 332: 17.4 | 17.6, 432: 18.7 | 18.2, 544: 19.8 | 18.6,
// 1232: 26.6 | 23.7.
constexpr uint32_t kWalkShareKeys = 352;
struct KeyRound {
    double d[16];
};
__device__ __forceinline__ void halves_to_f64(const uint4 &v, double *d) {
    const half8 h = as_half8(v);
#pragma unroll
    for (int j = 0; j < 8; j++) d[j] = double(float(h[j]));
}
// the sum over eight neighbouring lanes, in all of them
__device__ __forceinline__ double sum8_f64(double v) {
    v += dpp_f64<kDppQuadXor1>(v);
    v += dpp_f64<kDppQuadXor2>(v);
    return v + dpp_f64<kDppRowHalfMirror>(v);
}
__device__ bool walk_attention(const RmiWalkArgs &a, const WalkWords &at, gptr_word words, gptr_word mine, uint32_t idx, uint32_t step, uint32_t l,
                               uint32_t tag, uint4 *lds, WalkLds &sm) {
    // What follows from the thread and the position is worked out anew in every layer: the compiler would keep all of it in
    // registers across the layers, and spill.
    uint32_t tid = threadIdx.x;
    asm volatile("" : "+v"(tid), "+s"(step), "+s"(idx));
    constexpr uint32_t T = kWalkThreads, kPvp = 4, kPreK = 3, kPre = 6, kBatch = 8, kRound = T / 8;
    const uint32_t lane = tid & 63, hpk = a.n_head / a.n_head_kv;
    const uint32_t kvh = idx % a.n_head_kv, qh = (idx / a.n_head_kv) % hpk, pv_part = idx / a.n_head_kv / hpk;
    const uint32_t head = kvh * hpk + qh;
    const uint32_t n_keys = step + 1, n_cached = step, last_row = n_cached - 1;  // (step >= 1)
    const uint32_t n_pad = (n_keys + 63) / 64 * 64;
    double *wd = reinterpret_cast<double *>(lds);                       // [kWalkMaxKeys] softmax weights (f16 values)
    double *part = wd + kWalkMaxKeys;                                   // [waves][32]
    float *scores = reinterpret_cast<float *>(part + (T / 64) * 32);    // [kWalkMaxKeys + 32]
    const uint32_t row_u4 = a.kv_stride >> 3;
    const size_t layer_base = size_t(l) * a.capacity * a.kv_stride;
    const RmiWalkLayer w = table_entry(a.layers + l);
    // the cached keys whose scores this workgroup makes: [k_first, k_end)
    const bool share = n_keys >= kWalkShareKeys;
    const uint32_t quarter = (n_keys + 3) / 4, k_first = share ? pv_part * quarter : 0;
    const uint32_t k_end = share && k_first + quarter < n_cached ? k_first + quarter : n_cached;
    const uint32_t lane8 = tid & 7, key0 = k_first + (tid >> 3);
    const uint4 *kbase = reinterpret_cast<const uint4 *>(a.k_cache + layer_base + size_t(kvh) * 128) + lane8;
    auto key_at = [&](uint32_t t) { return kbase + __umul24(t < k_end ? t : last_row, row_u4); };
    // everything that does not depend on this position's q, k, v goes out before they are waited for
    float nw0 = 1.0f, nw1 = 1.0f, cos_a = 0.0f, sin_a = 0.0f;
    const float *norm = tid < 64 ? w.q_norm : w.k_norm;
    gptr_f32 nw = as_global<gptr_f32>(norm);
    if (tid < 128) {
        cos_a = a.cos_t[size_t(step) * 64 + lane];
        sin_a = a.sin_t[size_t(step) * 64 + lane];
        if (norm) {
            nw0 = nw[lane];
            nw1 = nw[lane + 64];
        }
    }
    KeyRound kd[kPreK];
    {
        uint4 raw[kPreK][2];
#pragma unroll
        for (uint32_t j = 0; j < kPreK; j++) {
            const uint4 *key = key_at(key0 + j * kRound);
            raw[j][0] = key[0];
            raw[j][1] = key[8];
        }
#pragma unroll
        for (uint32_t j = 0; j < kPreK; j++) {
            halves_to_f64(raw[j][0], kd[j].d);
            halves_to_f64(raw[j][1], kd[j].d + 8);
        }
    }
    constexpr uint32_t kDgLanes = 16 / kPvp, kSlices = T / kDgLanes;
    const uint32_t dg = tid % kDgLanes, sl = tid / kDgLanes;
    const uint32_t chunk = (n_keys + kSlices - 1) / kSlices;
    const uint32_t t_begin = sl * chunk, t_end = t_begin + chunk < n_keys ? t_begin + chunk : n_keys;
    const uint4 *vbase = reinterpret_cast<const uint4 *>(a.v_cache + layer_base + size_t(kvh) * 128 + pv_part * (128 / kPvp) + dg * 8);
    uint4 vp[kPre];
#pragma unroll
    for (uint32_t j = 0; j < kPre; j++) vp[j] = vbase[__umul24(t_begin + j < n_cached ? t_begin + j : last_row, row_u4)];
    uint4 kraw[2];  // the round behind the converted ones
    kraw[0] = key_at(key0 + kPreK * kRound)[0];
    kraw[1] = key_at(key0 + kPreK * kRound)[8];
    // keys and values have arrived before anything is stored: a later wait for them would be one for the stores, too
    for (const uint4 &r : kraw) asm volatile("" ::"v"(r.x));
#pragma unroll
    for (uint32_t j = 0; j < kPre; j++) asm volatile("" ::"v"(vp[j].x));
    if (tid < 192) {  // wave 0: q of this head, wave 1: the new k, wave 2: the new v; lane i owns (i, i + 64)
        const uint32_t which = tid >> 6;
        const uint32_t src = which == 0 ? head * 128 : a.n_head * 128 + (which == 1 ? kvh : a.n_head_kv + kvh) * 128;
        const gptr_word from[2] = {mine + at.qkv + src + lane, mine + at.qkv + src + lane + 64};
        uint32_t v[2];
        if (!words_wait<2>(from, tag, v, WalkBound{a.failed, a.spins})) sm.bad = 1;
        const float raw0 = __uint_as_float(v[0]), raw1 = __uint_as_float(v[1]);
        uint16_t h0, h1;
        if (which == 2) {
            h0 = rmi_f2h(raw0);
            h1 = rmi_f2h(raw1);
        } else {
            float x0 = raw0, x1 = raw1;
            if (norm) {
                const float q0 = raw0 * raw0, q1 = raw1 * raw1;
                double sum = double(q0);
                sum += double(q1);
                sum = wave_sum_f64(sum);
                const float mean_sq = float(sum / 128.0);
                const float sc = 1.0f / sqrtf(mean_sq + a.eps);
                x0 = (raw0 * sc) * nw0;
                x1 = (raw1 * sc) * nw1;
            }
            const float ta = x1 * -sin_a;
            const float tb = x1 * cos_a;
            h0 = rmi_f2h(__builtin_fmaf(x0, cos_a, ta));
            h1 = rmi_f2h(__builtin_fmaf(x0, sin_a, tb));
        }
        sm.new16[which][lane] = h0;
        sm.new16[which][lane + 64] = h1;
        if (which && qh == 0 && pv_part == 0) {  // the first query head of the key/value head fills the cache row, through to memory
            uint16_t *dst = (which == 1 ? a.k_cache : a.v_cache) + layer_base + size_t(step) * a.kv_stride + size_t(kvh) * 128;
            __hip_atomic_store(dst + lane, h0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(dst + lane + 64, h1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    __syncthreads();
    if (sm.bad) return false;
    double qd[16];
    halves_to_f64(reinterpret_cast<const uint4 *>(sm.new16[0])[lane8], qd);
    halves_to_f64(reinterpret_cast<const uint4 *>(sm.new16[0])[8 + lane8], qd + 8);
    const float kq_scale = 1.0f / sqrtf(128.0f);  // two f32 roundings, as the reference computes it
    float my_max = -INFINITY;
    gptr_word score_words = words + at.scores + head * kWalkMaxKeys;
    auto score = [&](const double *k, uint32_t t, bool live) {
        double s4[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int j = 0; j < 16; j++) s4[j & 3] = __builtin_fma(k[j], qd[j], s4[j & 3]);
        const float sc = float(sum8_f64((s4[0] + s4[1]) + (s4[2] + s4[3]))) * kq_scale;
        if (live && lane8 == 0) {
            if (share)
                word_store(score_words + t, __float_as_uint(sc), tag);
            else
                scores[t] = sc;
        }
        if (live) my_max = fmaxf(my_max, sc);
    };
    const uint32_t n_mine = k_first < k_end ? k_end - k_first : 0;
#pragma unroll
    for (uint32_t j = 0; j < kPreK; j++)
        if (j * kRound < n_mine) score(kd[j].d, key0 + j * kRound, key0 + j * kRound < k_end);
    for (uint32_t i0 = kPreK * kRound; i0 < n_mine; i0 += kRound) {
        KeyRound kr;
        halves_to_f64(kraw[0], kr.d);
        halves_to_f64(kraw[1], kr.d + 8);
        // the next round's keys are on their way while this one is summed (unconditional loads)
        kraw[0] = key_at(key0 + i0 + kRound)[0];
        kraw[1] = key_at(key0 + i0 + kRound)[8];
        score(kr.d, key0 + i0, key0 + i0 < k_end);
    }
    if (tid >= T - 64 && (!share || pv_part == kPvp - 1)) {  // this step's key, from LDS: the last wave
        KeyRound kr;
        halves_to_f64(reinterpret_cast<const uint4 *>(sm.new16[1])[lane8], kr.d);
        halves_to_f64(reinterpret_cast<const uint4 *>(sm.new16[1])[8 + lane8], kr.d + 8);
        score(kr.d, n_cached, lane < 8);
    }
    // the values, while the others' scores are on their way; this step's is in LDS
    const uint4 *v_new = reinterpret_cast<const uint4 *>(sm.new16[2]) + pv_part * kDgLanes + dg;
    KeyRound vd[kPre / 2];
#pragma unroll
    for (uint32_t j = 0; j < kPre; j++) {
        if (j < chunk) {
            if (t_begin + j == n_cached) vp[j] = *v_new;
            if (t_begin + j >= t_end) vp[j] = make_uint4(0, 0, 0, 0);  // not this slice's: zero times a weight of zero
            halves_to_f64(vp[j], vd[j / 2].d + 8 * (j & 1));
        }
    }
    constexpr int kMine = (kWalkMaxKeys + T - 1) / T;
    float e[kMine];  // of the keys tid, tid + T, ...
    if (share) {
        gptr_word from[kMine];
        uint32_t v[kMine];
#pragma unroll
        for (int j = 0; j < kMine; j++) from[j] = score_words + (j * T + tid < n_keys ? j * T + tid : n_keys - 1);
        if (!words_wait<kMine>(from, tag, v, WalkBound{a.failed, a.spins})) sm.bad = 1;
        my_max = -INFINITY;
#pragma unroll
        for (int j = 0; j < kMine; j++) {
            e[j] = __uint_as_float(v[j]);
            my_max = fmaxf(my_max, e[j]);
        }
    }
    my_max = wave_max_f32(my_max);
    if ((tid & 63) == 0) sm.max8[tid >> 6] = my_max;
    __syncthreads();
    if (sm.bad) return false;
    float max_val = sm.max8[0];
#pragma unroll
    for (uint32_t i = 1; i < T / 64; i++) max_val = fmaxf(max_val, sm.max8[i]);
#pragma unroll
    for (int j = 0; j < kMine; j++) {
        const uint32_t t = j * T + tid;
        if (t >= n_pad) break;
        if (!share) e[j] = scores[t];
        e[j] = t < n_keys ? rmi_expf_tab(e[j] - max_val, sm.exp_tab) : 0.0f;
        scores[t] = e[j];
    }
    __syncthreads();
    if (tid == 0) {  // the reference adds the weights one after the other in f32; the padding zeros change nothing
        float acc = 0.0f;
        constexpr int kAhead = 8;
        float4 b0[kAhead], b1[kAhead];
#pragma unroll
        for (int j = 0; j < kAhead; j++) b0[j] = reinterpret_cast<const float4 *>(scores)[j];
        for (uint32_t t = 0; t < n_pad; t += 8 * kAhead) {
#pragma unroll
            for (int j = 0; j < kAhead; j++) b1[j] = reinterpret_cast<const float4 *>(scores + t + 4 * kAhead)[j];
#pragma unroll
            for (int j = 0; j < kAhead; j++) {
                acc += b0[j].x;
                acc += b0[j].y;
                acc += b0[j].z;
                acc += b0[j].w;
            }
#pragma unroll
            for (int j = 0; j < kAhead; j++) b0[j] = reinterpret_cast<const float4 *>(scores + t + 8 * kAhead)[j];  // (32 floats of room)
#pragma unroll
            for (int j = 0; j < kAhead; j++) {
                acc += b1[j].x;
                acc += b1[j].y;
                acc += b1[j].z;
                acc += b1[j].w;
            }
        }
        sm.max8[0] = acc;
    }
    __syncthreads();
    const float total = sm.max8[0];
#pragma unroll
    for (int j = 0; j < kMine; j++) {
        const uint32_t t = j * T + tid;
        if (t >= n_pad) break;
        wd[t] = t < n_keys ? double(h2f(rmi_f2h(total > 0.0f ? e[j] / total : e[j]))) : 0.0;
    }
    __syncthreads();
    double acc[8];
#pragma unroll
    for (int j = 0; j < 8; j++) acc[j] = 0.0;
#pragma unroll
    for (uint32_t j = 0; j < kPre; j++) {
        if (j < chunk) {  // (at most 127 slices of ten keys, and five: inside wd)
            const double in_row = wd[t_begin + j], wt = t_begin + j < t_end ? in_row : 0.0;
#pragma unroll
            for (int d = 0; d < 8; d++) acc[d] = __builtin_fma(vd[j / 2].d[8 * (j & 1) + d], wt, acc[d]);
        }
    }
    auto add_value = [&](const uint4 &v, double wt) {
        const half8 vh = as_half8(v);
#pragma unroll
        for (int d = 0; d < 8; d++) acc[d] = __builtin_fma(double(float(vh[d])), wt, acc[d]);
    };
    if (t_begin + kPre < t_end) {  // longer slices: batches, the next one in flight while one is added
        uint4 cur[kBatch], nxt[kBatch];
#pragma unroll
        for (uint32_t j = 0; j < kBatch; j++) {
            const uint32_t t = t_begin + kPre + j;
            cur[j] = vbase[__umul24(t < n_cached ? t : last_row, row_u4)];
        }
        for (uint32_t t0 = t_begin + kPre; t0 < t_end; t0 += kBatch) {
#pragma unroll
            for (uint32_t j = 0; j < kBatch; j++) {
                const uint32_t t = t0 + kBatch + j;
                nxt[j] = vbase[__umul24(t < n_cached ? t : last_row, row_u4)];
            }
#pragma unroll
            for (uint32_t j = 0; j < kBatch; j++)
                if (t0 + j < t_end) add_value(t0 + j == n_cached ? *v_new : cur[j], wd[t0 + j]);
#pragma unroll
            for (uint32_t j = 0; j < kBatch; j++) cur[j] = nxt[j];
        }
    }
    {
        double u[2];
        pv_slices_sum<kDgLanes>(acc, u);
        if ((tid & 15) < kDgLanes) {
            double *dst = part + (tid >> 6) * 32 + dg * 8 + pv_dim_base(tid & 63);
            dst[0] = u[0];
            dst[1] = u[1];
        }
    }
    // the cache row is in memory before this workgroup's words say that the layer may go on (and so a later token may read it)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid < 64) {  // a dimension a lane, twice
        double o[T / 64];
#pragma unroll
        for (uint32_t wv = 0; wv < T / 64; wv++) o[wv] = part[wv * 32 + (lane & 31)];
        const float of = float(((o[0] + o[1]) + (o[2] + o[3])) + ((o[4] + o[5]) + (o[6] + o[7])));
        float sc;
        const uint32_t q = rmi_quantize_block32(of, a.rounding, &sc);
        block_store(words + at.att + (head * 4 + pv_part) * 9, at.n, q, sc, tag);
    }
    return true;
}

// Loads of a wave's N octets of a tile
template <int N>
__device__ __forceinline__ void octets_load(OctetRegs (&g)[N], const uint8_t *w, uint32_t tile, uint32_t n_oct, uint32_t first, uint32_t lane) {
    gptr_u4 t = as_global<gptr_u4>(w + size_t(tile) * n_oct * kOctetBytes);
#pragma unroll
    for (int i = 0; i < N; i++) load_octet(g[i], t + (lane >> 3), t + n_oct * 8 + lane, first + i);
}

// Four waves a tile of 4 N octets, staged in lds: the row's sum in the first wave (gemv_q8_0_deep_split_kernel)
template <int N>
__device__ __forceinline__ float tile_product(const OctetRegs (&g)[N], const uint4 *lds, uint32_t sub, uint32_t lane, float4 *hand) {
    const uint32_t L = lane & 7;
    if (sub != 0) octets_to_factors<N>(g, lds, 4 * N, sub * N, L, hand + (sub - 1) * N * 4 * 64 + lane);
    float acc = 0.0f;
    if (sub == 0) octets_fma_ahead<N>(acc, g, lds, L, 4 * N);
    __syncthreads();
    if (sub == 0) factors_sum<3 * N>(acc, hand + lane);
    return hsum8_lanes(acc);
}

// NE octets of the width; NO, ND octets a wave of the o and the down product (a quarter of theirs)
template <int NE, int NO, int ND>
__global__ __launch_bounds__(kWalkThreads) void qwen3_walk_kernel(RmiWalkArgs a) {
    extern __shared__ uint4 lds[];
    __shared__ WalkLds sm;
    const uint32_t tid = threadIdx.x, lane = tid & 63, r = lane >> 3, L = lane & 7;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr uint32_t n_embd = NE * 256;
    const WalkWords at = walk_words(n_embd, a.n_head, a.n_head_kv, a.n_ff, gridDim.x);
    gptr_word words = as_global<gptr_word>(a.words), mine = words + die_half() * at.n;
    if (tid == 0) sm.bad = 0;
    if (tid < 32) sm.exp_tab[tid] = kRmiExp2fTab[tid];
    __syncthreads();
    const uint32_t b = blockIdx.x;
    if (b < a.n_attn) {
        for (uint32_t i = 0; i < a.n_steps; i++) {
            const uint32_t tag = a.tag0 + 1 + i * (a.n_layer + 1);
            for (uint32_t l = 0; l < a.n_layer; l++) {
                if (!walk_attention(a, at, words, mine, b, a.step0 + i, l, tag + l, lds, sm)) return;
                __syncthreads();  // the words first: behind the other waves' keys and values they would wait for those
            }
            if (!walk_head<NE>(a, at, words, mine, tag + a.n_layer, a.keep_logits && i + 1 == a.n_steps, lds, sm)) return;
        }
        return;
    }
    if (b < a.n_attn + a.n_res) {
        const uint32_t idx = b - a.n_attn, sub = wave & 3, tile = idx * 2 + (wave >> 2), row = tile * 8 + r;
        float4 *hand = reinterpret_cast<float4 *>(lds + ND * 4 * 18) + (wave >> 2) * (3 * ND * 4 * 64);
        OctetRegs go[NO], gd[ND];
        float x = a.x[row];
        for (uint32_t i = 0; i < a.n_steps; i++) {
            const uint32_t tag = a.tag0 + 1 + i * (a.n_layer + 1), step = a.step0 + i;
            if (sub == 0 && L < 2) word_store(words + L * at.n + at.x + row, __float_as_uint(x), tag);
            octets_load<NO>(go, a.layers[0].o, tile, NO * 4, sub * NO, lane);
            octets_load<ND>(gd, a.layers[0].down, tile, ND * 4, sub * ND, lane);
            const uint32_t told = a.tok[step + 1];  // (the next token where the prompt still says it)
            for (uint32_t l = 0; l < a.n_layer; l++) {
                const RmiWalkLayer next = table_entry(a.layers + (l + 1 < a.n_layer ? l + 1 : l));
                if (!stage_quants<(NO * 4 * 72 + kWalkThreads - 1) / kWalkThreads>(mine + at.att, tag + l, NO * 4, a, lds, sm)) return;
                float y = tile_product<NO>(go, lds, sub, lane, hand);
                x = x + y;
                if (sub == 0 && L < 2) word_store(words + L * at.n + at.xm + row, __float_as_uint(x), tag + l);
                __syncthreads();  // the words first: behind other waves' weights they would wait for those
                octets_load<NO>(go, next.o, tile, NO * 4, sub * NO, lane);
                if (!stage_quants<(ND * 4 * 72 + kWalkThreads - 1) / kWalkThreads>(mine + at.h, tag + l, ND * 4, a, lds, sm)) return;
                y = tile_product<ND>(gd, lds, sub, lane, hand);
                x = x + y;
                if (sub == 0 && L < 2) word_store(words + L * at.n + at.x + row, __float_as_uint(x), tag + l + 1);
                __syncthreads();  // (x first, too)
                octets_load<ND>(gd, next.down, tile, ND * 4, sub * ND, lane);
            }
            __syncthreads();
            if (!walk_head<NE>(a, at, words, mine, tag + a.n_layer, a.keep_logits && i + 1 == a.n_steps, lds, sm)) return;
            // the next token, in every residual workgroup by itself, and the rows of its embedding
            const uint32_t n_wg = gridDim.x, g = tid < n_wg ? tid : n_wg - 1;
            const gptr_word top[4] = {mine + at.top + g * 4, mine + at.top + g * 4 + 1, mine + at.top + g * 4 + 2, mine + at.top + g * 4 + 3};
            uint32_t v[4];
            if (!words_wait<4>(top, tag + a.n_layer, v, WalkBound{a.failed, a.spins})) sm.bad = 1;
            Top m{__uint_as_float(v[0]), __uint_as_float(v[1]), v[2], v[3]};
            if (tid >= n_wg) m = Top{-INFINITY, -INFINITY, 0xffffffffu, 1u};
#pragma unroll
            for (int s = 32; s > 0; s >>= 1) {
                const Top other{__shfl_xor(m.best, s), __shfl_xor(m.second, s), uint32_t(__shfl_xor(int(m.id), s)),
                                uint32_t(__shfl_xor(int(m.finite), s))};
                m = top_merge(m, other);
            }
            if (lane == 0) sm.all_top[wave] = m;
            __syncthreads();
            if (sm.bad) return;
            m = sm.all_top[0];
#pragma unroll
            for (int s = 1; s < int(kWalkThreads / 64); s++) m = top_merge(m, sm.all_top[s]);
            uint32_t token = step + 1 >= a.n_prompt ? m.id : told;
            if (idx == 0 && tid == 0) {
                a.step_argmax[step] = m.id;
                a.step_top2[2 * step] = m.best;
                a.step_top2[2 * step + 1] = m.second;
                if (!m.finite) atomicAdd(a.nonfinite, 1u);
                if (step + 1 >= a.n_prompt) a.tok[step + 1] = m.id;
                static_cast<StepParams *>(a.sp)->step = step + 1;
            }
            if (token >= a.vocab) token = a.vocab - 1;  // never read outside the weight
            const uint8_t *et = a.embd + size_t(token >> 3) * NE * kOctetBytes;
            const uint32_t er = token & 7, eb = row >> 5, ek = row & 31;
            const uint16_t dh = *reinterpret_cast<const uint16_t *>(et + (eb >> 3) * 128 + er * 16 + (eb & 7) * 2);
            const int8_t q = *reinterpret_cast<const int8_t *>(et + size_t(NE) * 128 + size_t(eb >> 2) * 1024 + er * 128 + (ek >> 2) * 16 +
                                                               (eb & 3) * 4 + (ek & 3));
            x = h2f(dh) * float(int(q));
        }
        if (sub == 0 && L == 0) a.x[row] = x;
        return;
    }
    const uint32_t idx = b - a.n_attn - a.n_res;
    const uint32_t qkv_tiles = (a.n_head + 2 * a.n_head_kv) * 16, q_tile = idx + a.n_norm * wave;
    const bool q_live = q_tile < qkv_tiles;
    const uint32_t n_blk = a.n_ff / 32, up_tile0 = a.n_ff / 8;
    const uint32_t g_off = (wave < 4 ? 0u : up_tile0) + (wave & 3);
    const bool g_live = idx < n_blk;
    OctetRegs gq[NE], gg[NE];
    NormWeights<NE> wa, wf;
    for (uint32_t i = 0; i < a.n_steps; i++) {
        const uint32_t tag = a.tag0 + 1 + i * (a.n_layer + 1);
        // (waves without a tile load the first one's again: unconditional loads, in bounds)
        octets_load<NE>(gq, a.layers[0].qkv, q_live ? q_tile : 0, NE, 0, lane);
        octets_load<NE>(gg, a.layers[0].gu, g_off + (g_live ? idx : 0) * 4, NE, 0, lane);
        wa.load(a.layers[0].attn_norm);
        wf.load(a.layers[0].ffn_norm);
        for (uint32_t l = 0; l < a.n_layer; l++) {
            const RmiWalkLayer next = table_entry(a.layers + (l + 1 < a.n_layer ? l + 1 : l));
            if (!stage_norm<NE>(mine + at.x, tag + l, wa, a, lds, sm)) return;
            {
                float acc = 0.0f;
                octets_fma_ahead<NE>(acc, gq, lds, L);
                const float y = hsum8_lanes(acc);
                if (q_live && L < 2) word_store(words + L * at.n + at.qkv + q_tile * 8 + r, __float_as_uint(y), tag + l);
            }
            __syncthreads();  // every wave's words first: behind others' weights they would wait for those
            octets_load<NE>(gq, next.qkv, q_live ? q_tile : 0, NE, 0, lane);
            wa.load(next.attn_norm);
            if (!g_live) continue;
            if (!stage_norm<NE>(mine + at.xm, tag + l, wf, a, lds, sm)) return;
            for (uint32_t blk = idx; blk < n_blk; blk += a.n_norm) {
                if (blk != idx) octets_load<NE>(gg, a.layers[l].gu, g_off + blk * 4, NE, 0, lane);
                float acc = 0.0f;
                octets_fma_ahead<NE>(acc, gg, lds, L);
                const float y = hsum8_lanes(acc);
                if (L == 0) sm.gu[wave * 8 + r] = y;  // [0,32): gate rows of this block, [32,64): up rows
                __syncthreads();
                if (tid < 64) {
                    const uint32_t e = tid & 31;
                    const float gt = sm.gu[e], up = sm.gu[32 + e];
                    const float hv = up * (gt / (1.0f + rmi_expf_tab(-gt, sm.exp_tab)));
                    float sc;
                    const uint32_t q = rmi_quantize_block32(hv, a.rounding, &sc);
                    block_store(words + at.h + blk * 9, at.n, q, sc, tag + l);
                }
                if (blk + a.n_norm < n_blk) __syncthreads();  // gu is written again
            }
            __syncthreads();
            octets_load<NE>(gg, next.gu, g_off + idx * 4, NE, 0, lane);
            wf.load(next.ffn_norm);
        }
        __syncthreads();
        if (!walk_head<NE>(a, at, words, mine, tag + a.n_layer, a.keep_logits && i + 1 == a.n_steps, lds, sm)) return;
    }
}

struct WalkRoles {
    uint32_t attn, res, norm, all;
};
// attention takes four workgroups a head and the residual one for every sixteen rows; what is left norms
WalkRoles walk_roles(const RmiWalkShape &s) {
    WalkRoles r{};
    const uint32_t cus = uint32_t(rmi_device_cus());
    r.all = cus < kWalkThreads ? cus : kWalkThreads;
    r.attn = s.n_head * 4;
    r.res = s.n_embd / 16;
    r.norm = r.all > r.attn + r.res ? r.all - r.attn - r.res : 0;
    return r;
}

typedef void (*walk_kernel)(RmiWalkArgs);
struct WalkChoice {
    walk_kernel f;
    size_t lds;
};
constexpr size_t kWalkAttnLds = size_t(kWalkMaxKeys) * 8 + (kWalkThreads / 64) * 32 * 8 + (size_t(kWalkMaxKeys) + 32) * 4;
template <int NE, int NO, int ND>
WalkChoice walk_choice() {
    constexpr size_t staged = size_t(ND > NO ? ND : NO) * 4 * 288, hand = size_t(2) * 3 * ND * 4 * 64 * 16, norm = size_t(NE) * (288 + 1024);
    static_assert(ND >= NO, "the staged vector and what is handed over are sized by the down product");
    size_t lds = staged + hand;
    if (lds < norm) lds = norm;
    if (lds < kWalkAttnLds) lds = kWalkAttnLds;
    return WalkChoice{qwen3_walk_kernel<NE, NO, ND>, lds};
}
// The kernel for a width of NE octets: NO and ND follow from the o and the down product's rows, whose quarters are whole octets.
// us a token of eight layers and a vocabulary of 32768 by launches | walked, behind 100 keys and behind 1240, width, heads, n_ff:
//   512, 8, 1024 154 | 103, 247 | 171; 512, 16, 4096 180 | 119, 269 | 184; 1024, 8, 1024 170 | 112, 263 | 180;
//   1024, 8, 3072 165 | 120, 256 | 186; 1024, 16, 3072 180 | 125, 272 | 190; 1024, 16, 4096 198 | 127, 287 | 189.
// A workgroup of the norm role makes one block of 32 gate|up rows with weights that it has before the norm; all these sizes have as many
// norm workgroups as blocks.  Width 2048 with 16 heads and n_ff = 6144, as <8, 2, 6>, leaves 64 for 192 blocks, three rounds of which two
// wait for their weights: 294 | 305 behind 100 keys, 344 | 330 behind 700.  A product's rows that are no multiple of 1024 are not whole
// octets a wave, and 768 values of x not whole ones a thread.
template <int NE, int NO, int ND>
WalkChoice walk_choose_sizes(uint32_t n_attn, uint32_t n_ff) {
    if (n_attn == NO * 1024 && n_ff == ND * 1024) return walk_choice<NE, NO, ND>();
    if constexpr (ND < 4)
        return walk_choose_sizes<NE, NO, ND + 1>(n_attn, n_ff);
    else if constexpr (NO < 2)
        return walk_choose_sizes<NE, NO + 1, NO + 1>(n_attn, n_ff);
    else
        return WalkChoice{nullptr, 0};
}
WalkChoice walk_choose(const RmiWalkShape &s) {
    const uint32_t n_attn = s.n_head * 128;
    return s.n_embd == 512    ? walk_choose_sizes<2, 1, 1>(n_attn, s.n_ff)
           : s.n_embd == 1024 ? walk_choose_sizes<4, 1, 1>(n_attn, s.n_ff)
                              : WalkChoice{nullptr, 0};
}

}  // namespace

bool rmi_walk_qwen3_fits(const RmiWalkShape &s) {
    if (s.head_dim_k != 128 || s.head_dim_v != 128 || s.kv_stride != s.n_head_kv * 128) return false;
    const WalkChoice c = walk_choose(s);
    if (!c.f) return false;
    const WalkRoles r = walk_roles(s);
    if (r.norm == 0 || (s.n_head + 2 * s.n_head_kv) * 16 > r.norm * 8) return false;
    int coop = 0, per_cu = 0;
    if (hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, rmi_device()) != hipSuccess || !coop ||
        hipFuncSetAttribute(reinterpret_cast<const void *>(c.f), hipFuncAttributeMaxDynamicSharedMemorySize, int(c.lds)) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, c.f, int(kWalkThreads), c.lds) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return per_cu >= 1;
}

size_t rmi_walk_qwen3_words(const RmiWalkShape &s) {
    const WalkWords w = walk_words(s.n_embd, s.n_head, s.n_head_kv, s.n_ff, walk_roles(s).all);
    return w.scores + size_t(s.n_head) * kWalkMaxKeys;
}

int rmi_launch_walk_qwen3(const RmiWalkShape &s, RmiWalkArgs a, hipStream_t st) {
    if (a.step0 == 0 || a.n_steps == 0 || a.step0 + a.n_steps >= kWalkMaxKeys)
        return rmi_fail(RMI_HIP_E_INVALID, "%u positions from %u on are not the walk's", a.n_steps, a.step0);
    const WalkChoice c = walk_choose(s);
    const WalkRoles r = walk_roles(s);
    a.n_attn = r.attn;
    a.n_res = r.res;
    a.n_norm = r.norm;
    void *args[] = {&a};
    RMI_HIP_CHECK(hipLaunchCooperativeKernel(reinterpret_cast<const void *>(c.f), dim3(r.all), dim3(kWalkThreads), args, uint32_t(c.lds), st));
    return RMI_HIP_OK;
}
