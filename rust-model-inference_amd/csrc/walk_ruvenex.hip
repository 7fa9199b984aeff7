// A token of a Ruvenex session (bf16) by one cooperative launch that walks all layers: workgroups with roles that hand the
// vectors of a layer to one another, as in walk_qwen3.hip.
//
// By launches a layer of width 1024 is three dependent ones, 17 us, of which HBM needs 5.6 for its 38 MB.  Here, a workgroup of
// sixteen waves a compute unit,
//   an input workgroup   has six rows a wave of everything that reads h in registers (48 of them),
//   an output workgroup  ten rows of everything that ends in x (40), a piece of each a thread,
//   an attention workgroup (one a query head) the head's keys and values before its query is there,
//   a recurrence workgroup (one a head) its state,
// all of it loaded behind the layer before, so what a layer takes is the chain norm - product - mixer - product, and an exchange
// between each two.  The feed-forward's part of the last product is done while the mixers work.  Loads return in order: words that
// are asked for behind weights come behind them, so no workgroup asks for words soon after it has asked for weights (workgroups
// that held both products' weights found the feed-forward's words 5.7 us after their own product, in the place of 1.2).
//
// us a token by launches | walked, 28 layers of width 1024, the vocabulary's product and its copy apart: behind 140 keys 500 | 295,
// 420: 521 | 330; 4 layers behind 20: 88 | 77 (a cooperative launch costs some 15 more than another).  A layer, us behind 128 | 400 keys:
// 9.2 | 10.4, of that three exchanges 5.4 | 5.9 (x, which the input weights hold up behind few keys, 3.0 | 1.4; what the mixers read, for
// which keys and values have to be there, 1.1 | 3.5; their results 1.3 | 1.0), norm 0.5, the two products 0.8 to 1.1 each, mixers 1.6 | 2.2.
// A head's keys and values have to be in its workgroup's registers, so up to 511 keys; behind that, and for the first token, the single
// launches (a token of 28 layers and a vocabulary of 151936 then takes 560 us; walked it is 335 behind 110 keys, 384 behind 470).
//
// Words and tags as in walk_qwen3.hip.  A buffer is written again by a workgroup only behind words that depend on all its readers:
// everything that norms is behind the whole x of its layer, of which each row's owner has read the mixers' and the feed-forward's
// words and its gates of the layer before; mixers' words are behind everything that norms.  x itself is kept twice, by odd and even
// layers: a row of the next x does not depend on workgroups that make other rows' gates only, that of the one after next does.
// What crosses tokens (caches, history, state) crosses launches.
//
// Width 1024 only: a thread has whole values of x and a lane whole pieces of a row, which 512 and 1536 do not give, and 2048 would want 205
// output workgroups.  A wave's weights, six rows or a piece of ten, are what 128 registers hold beside the rest (of 48 bytes a lane that do
// not fit, addresses of the history, a mixer's wave reads some back in front of its wait for words): with those, 28-layer sizes of width
// 1024 and a feed-forward of 3072 are 256 workgroups, and more rows go by the single launches.
#include "walk_ruvenex.h"

#include "device_dense.h"
#include "device_walk.h"

namespace {

constexpr uint32_t T = 1024;
constexpr uint32_t kWidth = 1024, NQ = kWidth / 512;  // 16-byte pieces a lane of a row of the width
constexpr uint32_t kInRows = 6;    // of a wave, everything that reads h
constexpr uint32_t kOutRows = 10;  // of a workgroup, everything that ends in x
constexpr uint32_t kDim = 128;    // of every head
enum Seg { kSegQ, kSegK, kSegV, kSegGate, kSegRq, kSegRf, kSegRv, kSegG1, kSegG2, kSegUp, kSegs };

// where the exchange's vectors lie, in words; bf16 ones by two values a word
struct RvWords {
    uint32_t x[2], in, act, n;
};
__host__ __device__ inline RvWords rv_words(const RmiWalkRvShape &s) {
    RvWords w;
    w.x[0] = 0;
    w.x[1] = (s.width + 15) / 16 * 16;
    w.in = 2 * w.x[1];
    w.act = w.in + (s.n_rows + 15) / 16 * 16;
    w.n = w.act + s.k_pad / 2;
    return w;
}

struct RvLds {  // (arrays that are read by pieces of 16 bytes lie at such: a piece across two takes some 500 clocks a wave)
    alignas(16) float red[T / 64];
    alignas(16) float sum[T / 64];
    uint32_t bad;
    float gate[kOutRows][2];
    float part[T / 64][kOutRows];
    // attention
    alignas(16) rmi_bf16 q[kDim];
    alignas(16) rmi_bf16 k[kDim];
    alignas(16) rmi_bf16 v[kDim];
    alignas(16) rmi_bf16 weights[kWalkRvMaxKeys];
    float p[kWalkRvMaxKeys], own, groups[T / kDim][kDim];
    // recurrence
    float f[kDim], rq[kDim];
    alignas(16) float rv[kDim];
    alignas(16) float o[T / 32][kDim];
};

// the token's embedding: a launch of its own in front of a cooperative one is 14 us of a token of 411
__device__ __forceinline__ float embedded(const RmiWalkRvArgs &a, uint32_t col) {
    return a.embed.table ? embed_value<rmi_bf16>(a.embed, a.token, a.pos, col) : a.x[col];
}

struct RvCtx {
    const RmiWalkRvArgs &a;
    RvWords at;
    gptr_word words, mine;
    WalkBound bound;
};

// Sums over the wave of eight values a lane: lanes l with l & 15 < 4 hold that of value eighth(l), twice (copies (l >> 1) & 1).
// Halves and rows of sixteen are added by swaps that leave half as many values, then a row's lanes by DPP.
__device__ __forceinline__ uint32_t eighth(uint32_t lane) { return (lane & 1) + 2 * ((lane >> 4) & 1) + 4 * (lane >> 5); }
__device__ __forceinline__ float sums8(const float (&acc)[8]) {
    float v[4], u[2];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[k]), __float_as_uint(acc[k + 4]), false, false);
        v[k] = __uint_as_float(x[0]) + __uint_as_float(x[1]);
    }
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[k]), __float_as_uint(v[k + 2]), false, false);
        u[k] = __uint_as_float(x[0]) + __uint_as_float(x[1]);
        u[k] += dpp_f32<kDppQuadXor1>(u[k]);
        u[k] += dpp_f32<kDppQuadXor2>(u[k]);
        u[k] += dpp_f32<kDppRowHalfMirror>(u[k]);
        u[k] += dpp_f32<kDppRowMirror>(u[k]);
    }
    return threadIdx.x & 1 ? u[1] : u[0];
}

// two neighbouring lanes' values as bf16 to the word of the pair, both copies: lanes 2i of the lower half of `lanes` lanes the
// first, of the upper half (which hold the same values) the second
__device__ __forceinline__ void pair_store(const RvCtx &c, uint32_t word, float v, bool live, uint32_t copy, uint32_t tag) {
    const float other = dpp_f32<kDppQuadXor1>(v);
    if (live && (threadIdx.x & 1) == 0)
        word_store(c.words + copy * c.at.n + word, uint32_t(f32_to_bf16(v)) | (uint32_t(f32_to_bf16(other)) << 16), tag);
}

// ---- one query head
__device__ __forceinline__ bool walk_attention(const RvCtx &c, uint32_t of_head, uint32_t l, uint32_t tag, RvLds &sm) {
    const RmiWalkRvArgs &a = c.a;
    const RmiWalkRvShape &s = a.s;
    const RmiWalkRvLayer::Attn y = table_entry(&a.layers[l].attn);
    const uint32_t pos = a.pos;
    uint32_t tid = threadIdx.x, head = uint32_t(__builtin_amdgcn_readfirstlane(int(of_head)));
    asm volatile("" : "+v"(tid), "+s"(head));  // (what follows from them is worked out anew in every layer, not kept and spilled)
    const uint32_t lane = tid & 63, hpk = s.heads / s.kv_heads, kvh = head / hpk;
    const uint32_t channels = (s.heads + 2 * s.kv_heads) * kDim;
    // this thread's channel: of the query, the key, the value (128 threads each)
    const uint32_t which = tid >> 7, ch = tid & (kDim - 1);
    const uint32_t chan = which == 0 ? head * kDim + ch : which == 1 ? (s.heads + kvh) * kDim + ch : (s.heads + s.kv_heads + kvh) * kDim + ch;
    const bool has = which < 3, keeps = which == 0 || head % hpk == 0;  // the one of all workgroups that carries the channel on
    const uint32_t cc = has ? chan : 0;
    float hist[3], taps[4];
    gptr_f32 conv = as_global<gptr_f32>(y.conv) + size_t(cc) * s.taps, hin = as_global<gptr_f32>(a.now ? y.hist[1] : y.hist[0]);
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) {  // the last of four is the token's own; absent ones count for nothing
        const uint32_t off = 4 - s.taps, jj = j >= off ? j - off : 0;
        taps[j] = j >= off ? conv[jj] : 0.0f;
        if (j < 3) {
            const float h = hin[size_t(jj < s.taps - 1 ? jj : 0) * channels + cc];
            hist[j] = j >= off && pos + j >= 3 ? h : 0.0f;
        }
    }
    const uint32_t half = s.rot_dims / 2, ri = ch / 2;
    const bool turned = which < 2 && ri < half;
    const size_t ra = size_t(pos) * half + (turned ? ri : 0);
    const float cs = half ? as_global<gptr_f32>(y.cos_t)[ra] : 1.0f, sn = half ? as_global<gptr_f32>(y.sin_t)[ra] : 0.0f;
    // keys: eight lanes each, rounds of 128
    constexpr uint32_t kRound = T / 8, kRounds = kWalkRvMaxKeys / kRound, kGroups = T / kDim;
    const uint32_t lane8 = tid & 7, key0 = tid >> 3, last = pos - 1;
    gptr_u4 kc = as_global<gptr_u4>(y.k_cache) + size_t(kvh) * s.capacity * (kDim / 8) + lane8;
    u32x4 kr[kRounds][2];
#pragma unroll
    for (uint32_t j = 0; j < kRounds; j++) {
        if (j * kRound < pos) {
            const uint32_t t = key0 + j * kRound;
            kr[j][0] = kc[size_t(t < pos ? t : last) * (kDim / 8)];
            kr[j][1] = kc[size_t(t < pos ? t : last) * (kDim / 8) + 8];
        }
    }
    // values: a channel a thread, the blocks of 32 keys round the groups of threads; keys from pos on as zeros
    constexpr uint32_t kBlocks = kWalkRvMaxKeys / 32 / kGroups;
    gptr_u4 vc = as_global<gptr_u4>(y.v_cache) + size_t(kvh) * (s.capacity / 32) * kDim * 4 + ch * 4;
    u32x4 vr[kBlocks][4];
    const uint32_t group = uint32_t(__builtin_amdgcn_readfirstlane(int(which)));
#pragma unroll
    for (uint32_t j = 0; j < kBlocks; j++) {
        const uint32_t b = j * kGroups + group;
        if (b * 32 >= pos) break;
#pragma unroll
        for (uint32_t g = 0; g < 4; g++) vr[j][g] = vc[size_t(b) * kDim * 4 + g];
        if (b * 32 + 32 > pos) {  // the block that the token's own key lies in, or will
#pragma unroll
            for (uint32_t g = 0; g < 4; g++) {  // slots 8 g ..: keys 4 g .. 4 g + 3 and 16 + 4 g ..
                u32x4 v = vr[j][g];
#pragma unroll
                for (uint32_t d = 0; d < 4; d++) {
                    const uint32_t k = b * 32 + (d >> 1) * 16 + 4 * g + 2 * (d & 1);
                    const uint32_t word = v[d];
                    v[d] = k + 1 < pos ? word : k < pos ? word & 0xffffu : 0u;
                }
                vr[j][g] = v;
            }
        }
    }
    // keys and values have arrived before anything is stored: a later wait for them would be one for the stores, too
#pragma unroll
    for (uint32_t j = 0; j < kRounds; j++)
        if (j * kRound < pos) asm volatile("" ::"v"(kr[j][0]), "v"(kr[j][1]));
#pragma unroll
    for (uint32_t j = 0; j < kBlocks; j++)
        if ((j * kGroups + group) * 32 < pos) asm volatile("" ::"v"(vr[j][0]), "v"(vr[j][1]), "v"(vr[j][2]), "v"(vr[j][3]));
    // ---- the token's own channels
    const uint32_t in_row = which == 0 ? s.seg[kSegQ] + head * kDim + ch : which == 1 ? s.seg[kSegK] + kvh * kDim + ch : s.seg[kSegV] + kvh * kDim + ch;
    if (which < 4) {  // (the fourth group: the output's gate)
        const gptr_word from[1] = {c.mine + c.at.in + (has ? in_row : s.seg[kSegGate] + head)};
        uint32_t w[1];
        if (!words_wait<1>(from, tag, w, c.bound)) sm.bad = 1;
        const float u = __uint_as_float(w[0]);
        if (!has) {
            if (ch == 0) sm.own = u;
        } else {
            float z = 0.0f;
#pragma unroll
            for (uint32_t j = 0; j < 3; j++) z = __builtin_fmaf(taps[j], hist[j], z);
            z = __builtin_fmaf(taps[3], u, z);
            if (keeps) {
                float *ho = a.now ? y.hist[0] : y.hist[1];
                const uint32_t off = 4 - s.taps;
#pragma unroll
                for (uint32_t j = 1; j < 3; j++)
                    if (j > off) ho[size_t(j - 1 - off) * channels + chan] = hist[j];
                ho[size_t(s.taps - 2) * channels + chan] = u;
            }
            if (which < 2) {
                const float other = dpp_f32<kDppQuadXor1>(z);
                const float turn = ch & 1 ? __builtin_fmaf(z, cs, other * sn) : __builtin_fmaf(z, cs, -(other * sn));
                const rmi_bf16 r = f32_to_bf16(turned ? turn : z);
                (which == 0 ? sm.q : sm.k)[ch] = r;
                if (which == 1 && keeps) static_cast<rmi_bf16 *>(y.k_cache)[(size_t(kvh) * s.capacity + pos) * kDim + ch] = r;
            } else {
                const float sq = wave_sum_f32(z * z);
                if (lane == 0) sm.sum[(tid >> 6) & 1] = sq;
                hist[0] = z;
            }
        }
    }
    __syncthreads();
    if (sm.bad) return false;
    if (which == 2) {
        const float r = 1.0f / sqrtf((sm.sum[0] + sm.sum[1]) / float(kDim) + s.eps);
        const rmi_bf16 v = f32_to_bf16(hist[0] * r);
        sm.v[ch] = v;
        const uint32_t k = pos % 32;
        if (keeps)
            static_cast<rmi_bf16 *>(y.v_cache)[((size_t(kvh) * (s.capacity / 32) + pos / 32) * kDim + ch) * 32 + ((k >> 2) & 3) * 8 + (k >> 4) * 4 + (k & 3)] = v;
    }
    const u32x4 q0 = reinterpret_cast<const u32x4 *>(sm.q)[lane8], q1 = reinterpret_cast<const u32x4 *>(sm.q)[8 + lane8];
    float my_max = -INFINITY;
    auto sum8 = [](float v) {
        v += dpp_f32<kDppQuadXor1>(v);
        v += dpp_f32<kDppQuadXor2>(v);
        return v + dpp_f32<kDppRowHalfMirror>(v);
    };
#pragma unroll
    for (uint32_t j = 0; j < kRounds; j++) {
        if (j * kRound < pos) {
            const uint32_t t = key0 + j * kRound;
            const float z = sum8(dot_piece<rmi_bf16>(kr[j][1], q1, dot_piece<rmi_bf16>(kr[j][0], q0, 0.0f))) * s.attn_scale;
            if (t < pos) {
                if (lane8 == 0) sm.p[t] = z;
                my_max = fmaxf(my_max, z);
            }
        }
    }
    {  // the token's own key, in every wave
        const u32x4 k0 = reinterpret_cast<const u32x4 *>(sm.k)[lane8], k1 = reinterpret_cast<const u32x4 *>(sm.k)[8 + lane8];
        const float z = sum8(dot_piece<rmi_bf16>(k1, q1, dot_piece<rmi_bf16>(k0, q0, 0.0f))) * s.attn_scale;
        if (tid == 0) sm.p[pos] = z;
        my_max = fmaxf(my_max, z);
    }
    my_max = fmaxf(my_max, dpp_f32<kDppRowMirror>(my_max));
    my_max = fmaxf(my_max, __shfl_xor(my_max, 16));
    my_max = fmaxf(my_max, __shfl_xor(my_max, 32));
    if (lane == 0) sm.red[tid >> 6] = my_max;
    __syncthreads();
    float m = sm.red[0];
#pragma unroll
    for (uint32_t i = 1; i < T / 64; i++) m = fmaxf(m, sm.red[i]);
    // weights: one key a thread, in the values' order; the sum of the unrounded ones
    const float e = tid <= pos ? exp_t<rmi_bf16>(sm.p[tid] - m) : 0.0f;
    {
        const uint32_t k = tid & 31;
        if (tid < kWalkRvMaxKeys) sm.weights[(tid & ~31u) + ((k >> 2) & 3) * 8 + (k >> 4) * 4 + (k & 3)] = f32_to_bf16(tid < pos ? e : 0.0f);
        const float sum = wave_sum_f32(e);
        if (lane == 0) sm.sum[tid >> 6] = sum;
        if (tid == pos) sm.gate[0][0] = e;
    }
    __syncthreads();
    float total = 0.0f;
#pragma unroll
    for (uint32_t i = 0; i < T / 64; i++) total += sm.sum[i];
    float acc = which == 0 ? bf16_to_f32(sm.v[ch]) * bf16_to_f32(f32_to_bf16(sm.gate[0][0])) : 0.0f;
#pragma unroll
    for (uint32_t j = 0; j < kBlocks; j++) {
        if ((j * kGroups + group) * 32 >= pos) break;
        const u32x4 *pw = reinterpret_cast<const u32x4 *>(sm.weights) + (j * kGroups + group) * 4;
#pragma unroll
        for (uint32_t g = 0; g < 4; g++) acc = dot_piece<rmi_bf16>(vr[j][g], pw[g], acc);
    }
    sm.groups[which][ch] = acc;
    __syncthreads();
    if (tid < 2 * kDim) {
        float o = 0.0f;
#pragma unroll
        for (uint32_t i = 0; i < kGroups; i++) o += sm.groups[i][ch];
        o = o / total * sm.own;
        pair_store(c, c.at.act + (head * kDim + ch) / 2, o, true, tid >> 7, tag);
    }
    return true;
}

// ---- one head of the recurrence
__device__ __forceinline__ bool walk_recur(const RvCtx &c, uint32_t of_head, uint32_t l, uint32_t tag, RvLds &sm) {
    const RmiWalkRvArgs &a = c.a;
    const RmiWalkRvShape &s = a.s;
    const RmiWalkRvLayer::Recur y = table_entry(&a.layers[l].recur);
    uint32_t tid = threadIdx.x, head = uint32_t(__builtin_amdgcn_readfirstlane(int(of_head)));
    asm volatile("" : "+v"(tid), "+s"(head));
    constexpr uint32_t kSlices = T / 32, kPer = kDim / kSlices;  // state rows a thread
    const uint32_t quad = tid & 31, sl = tid >> 5, ch = tid & (kDim - 1), which = tid >> 7;
    gptr_u4 st = as_global<gptr_u4>(a.now ? y.state[1] : y.state[0]) + size_t(head) * kDim * (kDim / 4) + quad;
    f32x4 r[kPer];
#pragma unroll
    for (uint32_t j = 0; j < kPer; j++) r[j] = __builtin_bit_cast(f32x4, st[size_t(sl * kPer + j) * (kDim / 4)]);
    const float norm = as_global<gptr_f32>(y.norm)[ch];
    if (tid < 3 * kDim) {
        const gptr_word from[1] = {c.mine + c.at.in + (which == 0 ? s.seg[kSegRq] : which == 1 ? s.seg[kSegRf] : s.seg[kSegRv]) + head * kDim + ch};
        uint32_t w[1];
        if (!words_wait<1>(from, tag, w, c.bound)) sm.bad = 1;
        (which == 0 ? sm.rq : which == 1 ? sm.f : sm.rv)[ch] = __uint_as_float(w[0]);
    }
    __syncthreads();
    if (sm.bad) return false;
    const f32x4 v = reinterpret_cast<const f32x4 *>(sm.rv)[quad];
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (uint32_t j = 0; j < kPer; j++) {
        const float f = sm.f[sl * kPer + j], k = 1.0f - f, q = sm.rq[sl * kPer + j];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            r[j][e] = __builtin_fmaf(f, r[j][e], k * v[e]);
            o[e] = __builtin_fmaf(q, r[j][e], o[e]);
        }
    }
    *reinterpret_cast<f32x4 *>(&sm.o[sl][quad * 4]) = o;
    __syncthreads();
    float z = 0.0f;
#pragma unroll
    for (uint32_t i = 0; i < kSlices; i++) z += sm.o[i][ch];
    const float sq = wave_sum_f32(z * z);
    if ((tid & 63) == 0) sm.red[tid >> 6] = sq;
    __syncthreads();
    const float scale = 1.0f / sqrtf((sm.red[0] + sm.red[1]) / float(kDim) + s.eps);
    if (tid < 2 * kDim) pair_store(c, c.at.act + (s.k_attn + head * kDim + ch) / 2, z * scale * norm, true, which, tag);
    f32x4 *so = reinterpret_cast<f32x4 *>(a.now ? y.state[0] : y.state[1]) + size_t(head) * kDim * (kDim / 4) + quad;
#pragma unroll
    for (uint32_t j = 0; j < kPer; j++) so[size_t(sl * kPer + j) * (kDim / 4)] = r[j];
    return true;
}

// ---- everything that reads h: kInRows rows a wave
__device__ __forceinline__ void walk_input(const RvCtx &c, uint32_t idx, RvLds &sm, u32x4 *h) {
    const RmiWalkRvArgs &a = c.a;
    const RmiWalkRvShape &s = a.s;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = uint32_t(__builtin_amdgcn_readfirstlane(int(tid >> 6)));
    const uint32_t row0 = (idx * (T / 64) + wave) * kInRows, row = row0 + eighth(lane), copy = (lane >> 1) & 1;
    const bool live = row0 < s.n_rows, stores = eighth(lane) < kInRows && row < s.n_rows && (lane & 15) < 4;
    // this lane's row: its segment (a wave's rows may lie in two)
    uint32_t seg = 0, seg0 = 0;
#pragma unroll
    for (uint32_t i = 1; i < kSegs; i++) {
        seg = row >= s.seg[i] ? i : seg;
        seg0 = row >= s.seg[i] ? s.seg[i] : seg0;
    }
    const uint32_t in_seg = stores ? row - seg0 : 0;
    const uint32_t act_of = seg == kSegRq ? kActSilu : seg == kSegRf ? kActForgetGate : seg == kSegUp ? kActGeluTanh : seg == kSegGate || seg == kSegG1 || seg == kSegG2 ? kActSigmoid : kActNone;
    constexpr uint32_t kX = NQ * 512 / T;  // values of x a thread
    static_assert(kX >= 1, "whole values a thread");
    u32x4 wi[kInRows][NQ];
    float bias, lower, wn[kX];
    auto load = [&](uint32_t l) {
        const RmiWalkRvLayer::In y = table_entry(&a.layers[l].in);
        gptr_u4 w = as_global<gptr_u4>(static_cast<const rmi_bf16 *>(y.w) + size_t(live ? row0 : 0) * s.in_ld) + lane;
#pragma unroll
        for (uint32_t r = 0; r < kInRows; r++)
#pragma unroll
            for (uint32_t q = 0; q < NQ; q++) wi[r][q] = __builtin_nontemporal_load(w + (row0 + r < s.n_rows ? size_t(r) : 0) * (s.in_ld / 8) + q * 64);
        const float *bp = seg == kSegRf ? y.f_bias : seg == kSegG1 ? y.b1 : seg == kSegG2 ? y.b2 : nullptr;
        bias = as_global<gptr_f32>(bp ? bp : y.norm)[bp ? in_seg : 0];
        if (!bp) bias = 0.0f;
        lower = as_global<gptr_f32>(seg == kSegRf ? y.lower : y.norm)[seg == kSegRf ? in_seg : 0];
#pragma unroll
        for (uint32_t j = 0; j < kX; j++) wn[j] = tid + j * T < s.width ? as_global<gptr_f32>(y.norm)[tid + j * T] : 0.0f;
    };
    load(0);
    for (uint32_t l = 0; l < s.n_layer; l++) {
        const uint32_t tag = a.tag0 + 1 + l;
        float x[kX], sq = 0.0f;
        if (l == 0) {
#pragma unroll
            for (uint32_t j = 0; j < kX; j++) x[j] = tid + j * T < s.width ? embedded(a, tid + j * T) : 0.0f;
        } else {
            gptr_word from[kX];
            uint32_t w[kX];
#pragma unroll
            for (uint32_t j = 0; j < kX; j++) from[j] = c.mine + (l & 1 ? c.at.x[1] : c.at.x[0]) + (tid + j * T < s.width ? tid + j * T : 0);
            if (!words_wait<kX>(from, tag, w, c.bound)) sm.bad = 1;
#pragma unroll
            for (uint32_t j = 0; j < kX; j++) x[j] = tid + j * T < s.width ? __uint_as_float(w[j]) : 0.0f;
        }
#pragma unroll
        for (uint32_t j = 0; j < kX; j++) sq = __builtin_fmaf(x[j], x[j], sq);
        sq = wave_sum_f32(sq);
        if (lane == 0) sm.red[wave] = sq;
        __syncthreads();
        if (sm.bad) return;
        float total = 0.0f;
#pragma unroll
        for (uint32_t i = 0; i < T / 64; i++) total += sm.red[i];
        const float scale = 1.0f / sqrtf(total / float(s.width) + s.eps);
#pragma unroll
        for (uint32_t j = 0; j < kX; j++) reinterpret_cast<rmi_bf16 *>(h)[tid + j * T] = f32_to_bf16(x[j] * scale * wn[j]);
        __syncthreads();
        float acc[8];
#pragma unroll
        for (uint32_t r = 0; r < 8; r++) acc[r] = 0.0f;
#pragma unroll
        for (uint32_t q = 0; q < NQ; q++) {
            const u32x4 hv = h[q * 64 + lane];
#pragma unroll
            for (uint32_t r = 0; r < kInRows; r++) acc[r] = dot_piece<rmi_bf16>(wi[r][q], hv, acc[r]);
        }
        const float o = apply_act<rmi_bf16>(act_of, sums8(acc), bias, lower);
        pair_store(c, c.at.act + (s.k_recur + in_seg) / 2, o, stores && seg == kSegUp, copy, tag);
        if (stores && seg != kSegUp)
            word_store(c.words + copy * c.at.n + c.at.in + row, __float_as_uint(o), tag);
        __syncthreads();  // every wave's words are on their way: behind the first ones' weights they would wait for those
        if (l + 1 < s.n_layer) load(l + 1);
    }
}

// ---- everything that ends in x: kOutRows rows a workgroup, of each the piece tid a thread
__device__ __forceinline__ void walk_output(const RvCtx &c, uint32_t idx, RvLds &sm, u32x4 *act) {
    const RmiWalkRvArgs &a = c.a;
    const RmiWalkRvShape &s = a.s;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = uint32_t(__builtin_amdgcn_readfirstlane(int(tid >> 6)));
    const uint32_t out0 = idx * kOutRows, pieces = s.k_pad / 8, up0 = s.k_recur / 2, n_act = s.k_pad / 2;  // (act in words)
    u32x4 wo[kOutRows];
    auto load = [&](uint32_t l) {
        gptr_u4 w = as_global<gptr_u4>(table_entry(&a.layers[l].out).w) + (tid < pieces ? tid : pieces - 1);
#pragma unroll
        for (uint32_t r = 0; r < kOutRows; r++)
            wo[r] = __builtin_nontemporal_load(w + size_t(out0 + r < s.width ? out0 + r : s.width - 1) * (s.out_ld / 8));
    };
    const uint32_t part_of = tid * 8 < s.k_attn ? 0u : tid * 8 < s.k_recur ? 1u : 2u;
    const float part_scale = part_of == 0 ? s.left_scale : part_of == 1 ? s.right_scale : 1.0f;
    const bool has = tid < pieces;
    const uint32_t my_row = out0 + (lane & 15);  // of lanes whose lane & 15 is below kOutRows
    float x_own = embedded(a, my_row < s.width ? my_row : s.width - 1);
    load(0);
    // words of act to LDS
    auto stage = [&](uint32_t first, uint32_t n, uint32_t tag) {
        constexpr uint32_t kMost = 4;
        const gptr_word at = c.mine + c.at.act + first;
        uint32_t w[kMost];
        if (n > 2 * T) {
            gptr_word from[kMost];
#pragma unroll
            for (uint32_t j = 0; j < kMost; j++) from[j] = at + (j * T + tid < n ? j * T + tid : 0);
            if (!words_wait<kMost>(from, tag, w, c.bound)) sm.bad = 1;
        } else {
            gptr_word from[2];
            uint32_t v[2];
#pragma unroll
            for (uint32_t j = 0; j < 2; j++) from[j] = at + (j * T + tid < n ? j * T + tid : 0);
            if (!words_wait<2>(from, tag, v, c.bound)) sm.bad = 1;
            w[0] = v[0], w[1] = v[1], w[2] = w[3] = 0;
        }
#pragma unroll
        for (uint32_t j = 0; j < kMost; j++)
            if (j * T + tid < n) reinterpret_cast<uint32_t *>(act)[first + j * T + tid] = w[j];
    };
    for (uint32_t l = 0; l < s.n_layer; l++) {
        const uint32_t tag = a.tag0 + 1 + l;
        // the feed-forward's activations and the gates, while the mixers work
        stage(up0, n_act - up0, tag);
        if (tid < 64) {
            const uint32_t r = (lane & 15) < kOutRows ? lane & 15 : 0, g = (lane >> 4) & 1, row = out0 + r < s.width ? out0 + r : s.width - 1;
            const gptr_word gate[1] = {c.mine + c.at.in + (g ? s.seg[kSegG2] : s.seg[kSegG1]) + row};
            uint32_t v[1];
            if (!words_wait<1>(gate, tag, v, c.bound)) sm.bad = 1;
            if (lane < 32 && (lane & 15) < kOutRows) sm.gate[r][g] = __uint_as_float(v[0]);
        }
        __syncthreads();
        if (sm.bad) return;
        float acc[kOutRows];
#pragma unroll
        for (uint32_t r = 0; r < kOutRows; r++) acc[r] = 0.0f;
        auto product = [&] {
            const u32x4 av = act[tid];
#pragma unroll
            for (uint32_t r = 0; r < kOutRows; r++) acc[r] = sm.gate[r][part_of == 2 ? 1 : 0] * part_scale * dot_piece<rmi_bf16>(wo[r], av, 0.0f);
        };
        if (has && part_of == 2) product();
        stage(0, up0, tag);
        __syncthreads();
        if (sm.bad) return;
        if (has && part_of != 2) product();
        static_assert(kOutRows == 10, "eight sums and two");
        const float sum = sums8(reinterpret_cast<const float(&)[8]>(acc)), sum8 = wave_sum_f32(acc[8]), sum9 = wave_sum_f32(acc[9]);
        if ((lane & 15) < 2) sm.part[wave][eighth(lane)] = sum;
        if (lane < 2) sm.part[wave][8 + lane] = lane ? sum9 : sum8;
        __syncthreads();
        if (tid < 64) {
            float z = 0.0f;
#pragma unroll
            for (uint32_t w = 0; w < T / 64; w++) z += sm.part[w][(lane & 15) < kOutRows ? lane & 15 : 0];
            x_own += z;
            if (lane < 32 && (lane & 15) < kOutRows && my_row < s.width && (l + 1 < s.n_layer || a.head))
                word_store(c.words + (lane >> 4) * c.at.n + (l & 1 ? c.at.x[0] : c.at.x[1]) + my_row, __float_as_uint(x_own), tag + 1);
        }
        __syncthreads();  // (x first, too)
        if (l + 1 < s.n_layer) load(l + 1);
    }
    if (tid < kOutRows && my_row < s.width) a.x[my_row] = x_own;
}

// ---- the vocabulary: every workgroup, eight rows a wave at a time.  A launch behind a cooperative one begins 11 us after it; here the first
// rows are asked for in front of the last layer's vector, and a row's place in the registers takes the next one as soon as it is multiplied.
__device__ __forceinline__ void walk_head(const RvCtx &c, RvLds &sm, u32x4 *h) {
    const RmiWalkRvArgs &a = c.a;
    const RmiWalkRvShape &s = a.s;
    constexpr uint32_t kRows = 8, kX = NQ * 512 / T;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = uint32_t(__builtin_amdgcn_readfirstlane(int(tid >> 6)));
    const uint32_t units = (a.vocab + kRows - 1) / kRows, step = gridDim.x * (T / 64);
    uint32_t unit = blockIdx.x * (T / 64) + wave;
    const gptr_u4 rows = as_global<gptr_u4>(a.head) + lane;
    u32x4 w[kRows][NQ];
    auto load = [&](uint32_t u, uint32_t r) {  // (rows are padded to sixteen)
        const gptr_u4 at = rows + size_t((u < units ? u : units - 1) * kRows + r) * (s.in_ld / 8);
#pragma unroll
        for (uint32_t q = 0; q < NQ; q++) w[r][q] = __builtin_nontemporal_load(at + q * 64);
    };
#pragma unroll
    for (uint32_t r = 0; r < kRows; r++) load(unit, r);
    float x[kX], wn[kX], sq = 0.0f;
    gptr_word from[kX];
    uint32_t v[kX];
#pragma unroll
    for (uint32_t j = 0; j < kX; j++) {
        wn[j] = as_global<gptr_f32>(a.head_norm)[tid + j * T];
        from[j] = c.mine + (s.n_layer & 1 ? c.at.x[1] : c.at.x[0]) + tid + j * T;
    }
    if (!words_wait<kX>(from, a.tag0 + 1 + s.n_layer, v, c.bound)) sm.bad = 1;
#pragma unroll
    for (uint32_t j = 0; j < kX; j++) {
        x[j] = __uint_as_float(v[j]);
        sq = __builtin_fmaf(x[j], x[j], sq);
    }
    sq = wave_sum_f32(sq);
    if (lane == 0) sm.red[wave] = sq;
    __syncthreads();
    if (sm.bad) return;
    float total = 0.0f;
#pragma unroll
    for (uint32_t i = 0; i < T / 64; i++) total += sm.red[i];
    const float scale = 1.0f / sqrtf(total / float(s.width) + s.eps);
#pragma unroll
    for (uint32_t j = 0; j < kX; j++) reinterpret_cast<rmi_bf16 *>(h)[tid + j * T] = f32_to_bf16(x[j] * scale * wn[j]);
    __syncthreads();
    u32x4 hv[NQ];
#pragma unroll
    for (uint32_t q = 0; q < NQ; q++) hv[q] = h[q * 64 + lane];
    for (; unit < units; unit += step) {
        float acc[kRows];
#pragma unroll
        for (uint32_t r = 0; r < kRows; r++) {
            acc[r] = 0.0f;
#pragma unroll
            for (uint32_t q = 0; q < NQ; q++) acc[r] = dot_piece<rmi_bf16>(w[r][q], hv[q], acc[r]);
            load(unit + step, r);
        }
        const float sum = sums8(acc);
        const uint32_t row = unit * kRows + eighth(lane);
        if ((lane & 15) < 2 && row < a.vocab) a.logits[row] = sum;
    }
}

__global__ __launch_bounds__(T) void ruvenex_walk_kernel(RmiWalkRvArgs a) {
    __shared__ RvLds sm;
    __shared__ u32x4 staged[T];  // the normed stream, or what the last product reads
    const RmiWalkRvShape &s = a.s;
    const RvWords at = rv_words(s);
    gptr_word words = as_global<gptr_word>(a.words);
    const RvCtx c{a, at, words, words + die_half() * at.n, WalkBound{a.failed, a.spins}};
    if (threadIdx.x == 0) sm.bad = 0;
    if (a.embed.table && blockIdx.x == 0 && threadIdx.x == 0) *a.tok_out = a.token;
    __syncthreads();
    const uint32_t b = blockIdx.x, n_mix = s.heads + s.recur_heads;
    if (b < n_mix) {
        for (uint32_t l = 0; l < s.n_layer; l++) {
            // (a key/value head's workgroups on one XCD, if it has eight of them)
            const uint32_t head = b % s.kv_heads * (s.heads / s.kv_heads) + b / s.kv_heads;
            const bool ok = b < s.heads ? walk_attention(c, head, l, a.tag0 + 1 + l, sm) : walk_recur(c, b - s.heads, l, a.tag0 + 1 + l, sm);
            if (!ok) return;
            __syncthreads();
        }
    } else if (b < n_mix + a.n_output) {
        walk_output(c, b - n_mix, sm, staged);
    } else {
        walk_input(c, b - n_mix - a.n_output, sm, staged);
    }
    if (a.head) {
        __syncthreads();
        const bool bad = sm.bad != 0;
        __syncthreads();  // (nobody gives up a wait before everybody has read it)
        if (!bad) walk_head(c, sm, staged);
    }
}

struct Roles {
    uint32_t mixers, output, input;
    uint32_t all() const { return mixers + output + input; }
};
Roles roles_of(const RmiWalkRvShape &s) {
    return Roles{s.heads + s.recur_heads, (s.width + kOutRows - 1) / kOutRows, (s.n_rows + T / 64 * kInRows - 1) / (T / 64 * kInRows)};
}

}  // namespace

bool rmi_walk_ruvenex_fits(const RmiWalkRvShape &s) {
    // The embedding lies where the last layer's x goes.  With a layer between, whose x all of the last one depends on, everybody has read it by
    // then; with one layer an input workgroup that makes other rows' gates only may not have.
    if (s.n_layer < 2) return false;
    if (s.k_in != kWidth || s.width != s.k_in || s.k_pad / 8 > T || roles_of(s).all() > uint32_t(rmi_device_cus())) return false;
    if (s.k_attn != s.heads * kDim || s.k_recur - s.k_attn != s.recur_heads * kDim || s.taps > 4 || s.taps < 2 || s.heads % s.kv_heads) return false;
    if (s.seg[kSegs] - s.seg[kSegUp] != s.k_pad - s.k_recur) return false;
    int coop = 0, per_cu = 0;
    if (hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, rmi_device()) != hipSuccess || !coop ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, ruvenex_walk_kernel, int(T), 0) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return per_cu >= 1;
}

size_t rmi_walk_ruvenex_words(const RmiWalkRvShape &s) { return 2 * size_t(rv_words(s).n); }

int rmi_launch_walk_ruvenex(RmiWalkRvArgs a, hipStream_t st) {
    if (a.pos == 0 || a.pos >= kWalkRvMaxKeys) return rmi_fail(RMI_HIP_E_INVALID, "position %u is not the walk's", a.pos);
    const Roles r = roles_of(a.s);
    a.n_output = r.output;
    void *args[] = {&a};
    RMI_HIP_CHECK(hipLaunchCooperativeKernel(reinterpret_cast<const void *>(ruvenex_walk_kernel), dim3(r.all()), dim3(T), args, 0, st));
    return RMI_HIP_OK;
}
