// A token of a Vogizen session by one cooperative launch that walks all layer runs: workgroups with roles that hand a run's vectors to
// one another, as in walk_qwen3.hip and walk_ruvenex.hip.
//
// By launches a run of width 2048 is seven dependent ones with a delta rule, eight with latent attention, 52 us in bf16 and 66 in f32,
// of which HBM needs 17 and 33 for 117 and 218 MB.  Here a workgroup of sixteen waves a compute unit is
//   stream   (six a kilobyte of a row's 64: 192 or 96) what reads the stream first, the latents' up-projections, the feed-forward, the
//            loop's product; four rows of the feed-forward a wave
//   chain    (64) a mixer (a head of the delta rule, a quarter of a head's keys), the output, the token's gate, its projection
// A phase's weights are asked for right behind the words of the phase before, so that they arrive while the vector is still being
// made; a run's weights are more than the chip's registers hold (as they are not in walk_ruvenex.hip), so every workgroup of the stream
// takes part in every large product.  Loads return in order: words that are asked for behind weights come behind them.
//
// us a token by launches | walked, without the vocabulary's product: eight runs of width 2048 behind 300 keys, bf16 418 | 278, f32 562 |
// 446; 28 of width 1024 behind 60, bf16 985 | 600 to 630, f32 1099 | 770 to 830.  A run with a delta rule then is 27 us in bf16 and 47 in
// f32, where memory is busy most of the time (4.6 TB/s; a phase's loads start 2 us behind the words before them).  Of the 19.4 of width
// 1024 in bf16 products are 3.9 and the mixer 2.9, norms 1.5, the rest is exchanges of 1.2 to 2.4, seven of them.
//
// Words and tags as in walk_qwen3.hip.  All of a run's vectors are kept twice, by odd and even runs: a workgroup writes one again only
// after it has waited for words of the run between, which depend on every other workgroup's: the feed-forward's on all of the stream's,
// the projection's on all of the chain's.  A wait that is given up leaves garbage in vectors but in no address: the workgroup ends behind
// the run, the launch is marked as failed, and the session takes the token again by single launches.
//
// Position 0 and positions that see more than 1024 keys go by the single launches.
#include "walk_vogizen.h"

#include <type_traits>

#include "device_dense.h"
#include "device_walk.h"

namespace {

constexpr uint32_t T = 1024;       // threads
constexpr uint32_t kWaves = T / 64;
constexpr uint32_t kHeads = 16, kDim = 128, kValues = kHeads * kDim;  // of either mixer
constexpr uint32_t kChain = 64;    // workgroups of mixers, output, gate and projection
constexpr uint32_t kParts = kChain / kHeads;  // of a head's keys
constexpr uint32_t kPartBlocks = (kWalkVgKeys / kKeyBlock + 1 + kParts - 1) / kParts;  // of a part, at most
constexpr uint32_t kPartWords = kDim + 2;

// Sizes that follow from the element type and the width.
template <typename El, uint32_t W>
struct Vg {
    static constexpr uint32_t E = sizeof(El), NP = W * E / 1024;  // 16-byte pieces a lane of a row of W
    static constexpr uint32_t kHeld = 16, B = kHeld / NP;         // pieces a lane holds, and rows they are
    static constexpr uint32_t kFf = 3 * W;
    static constexpr uint32_t kStream = 2 * kFf / 64;             // workgroups with the large products: four rows of the feed-forward a wave
    static constexpr uint32_t KX = W / T;                         // values of the stream a thread
    static constexpr uint32_t kDownRows = (W + kStream - 1) / kStream;
    static constexpr uint32_t kInUnits = W == 1024 ? 6 : 3;       // rows a wave of what reads the stream first, at most
    static constexpr uint32_t kMaxQ = W == 1024 ? 768 : 1024, kMaxKv = W / 4;
    static constexpr uint32_t NPQ = (kMaxQ * E + 1023) / 1024, NPK = (kMaxKv * E + 1023) / 1024;
    static constexpr uint32_t kUpQ = (kValues + kStream - 1) / kStream, kUpKv = (2 * kValues + kStream - 1) / kStream;  // rows a workgroup
    static constexpr uint32_t kUpQUnits = (kUpQ + kWaves - 1) / kWaves, kUpKvUnits = (kUpKv + kWaves - 1) / kWaves;
    static constexpr uint32_t kRowPieces = W * E / 16;
    // Of the feed-forward's last product, a wave's thirds of a row: those that wait in LDS since the first is worked on, where registers
    // hold less than three, and in registers.  (All in LDS, where there is room: bf16 of 2048 307 us a token in the place of 276, for the words
    // of the first come behind them; f32 of 1024 809 and 772.)
    static constexpr uint32_t kDownAhead = NP * 3 > kHeld ? 1 : 0, kDownHeld = 3 - kDownAhead;
    static_assert(kDownHeld <= B, "what is not in LDS");
    static constexpr uint32_t kOwn = W / kChain, kOwnUnits = kOwn / kWaves, NPO = kValues * E / 1024;  // rows of the output a chain workgroup, a wave
    static constexpr bool kOutAhead = E == 2;  // asked for a run ahead, while the feed-forward is worked on: f32 keys and values leave no room
    static_assert(NP * B == kHeld && kUpQUnits * NPQ + kUpKvUnits * NPK <= kHeld, "what a lane holds");
    static_assert((kDownRows * 3 + kWaves - 1) / kWaves == 3, "units of the last product");
};

// where the vectors of a run lie, in words; those that products read as operands by sizeof(El) / 4 words a value
struct VgWords {
    uint32_t in, up, part, act, xa, ff, xb, side, y, xl, n;
};
__host__ __device__ inline VgWords vg_words(const RmiWalkVgShape &s) {
    VgWords w;
    uint32_t at = 0;
    auto take = [&](uint32_t n) {
        const uint32_t a = at;
        at += (n + 15) / 16 * 16;
        return a;
    };
    w.in = take(s.delta_rows > s.latent_rows ? s.delta_rows : s.latent_rows);
    w.up = take(3 * kValues);
    w.part = take(kChain * kPartWords);
    w.act = take(kValues * s.elem_bytes / 4);
    w.xa = take(s.width);
    w.ff = take(3 * s.width * s.elem_bytes / 4);
    w.xb = take(s.width);
    w.side = take(s.side);
    w.y = take(s.width);
    w.xl = take(s.width);
    w.n = at;
    return w;
}

template <typename El, uint32_t W>
struct VgLds {
    alignas(16) float red[4][kWaves];
    float2 stats[kWaves];
    uint32_t bad;
    union {
        struct {
            float part[3 * Vg<El, W>::kDownRows], own[Vg<El, W>::kDownRows];
            alignas(16) u32x4 down[Vg<El, W>::kDownAhead ? kWaves * Vg<El, W>::kRowPieces : 1];
        } s;
        struct {
            float own[Vg<El, W>::kOwn], gate[kWaves];
            alignas(16) float f[5][kDim];   // q, k, v, gate; u
            alignas(16) float part[2][T / 32][kDim];
            float ba[2], sums[2][kDim];
            alignas(16) El q[kDim], k[kDim];
            float v[kDim];
            float p[kPartBlocks * kKeyBlock];
            alignas(16) El weights[(kPartBlocks + 1) * kKeyBlock];
            float own_p, own_e, groups[T / kDim][kDim];
        } c;
    };
};

struct VgCtx {
    const RmiWalkVgArgs &a;
    VgWords at;
    gptr_word words, mine;
    WalkBound bound;
    // a run's vectors: where the workgroup reads them, where a copy is stored
    __device__ __forceinline__ gptr_word from(uint32_t run) const { return mine + (run & 1) * at.n; }
    __device__ __forceinline__ gptr_word to(uint32_t run, uint32_t copy) const { return words + (copy * 2 + (run & 1)) * at.n; }
    __device__ __forceinline__ uint32_t tag(uint32_t run) const { return a.tag0 + 1 + run; }
};

// the sum of a row of sixteen lanes, in each of them
__device__ __forceinline__ float row_sum(float v) {
    v += dpp_f32<kDppQuadXor1>(v);
    v += dpp_f32<kDppQuadXor2>(v);
    v += dpp_f32<kDppRowHalfMirror>(v);
    return v + dpp_f32<kDppRowMirror>(v);
}
// sum over the workgroup; `red` is not written again before another barrier
static_assert(kWaves == 16, "a wave's sum a lane of a row");
__device__ __forceinline__ float group_sum(float v, float *red) {
    v = wave_sum_f32(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return row_sum(red[threadIdx.x & 15]);
}

// words base + tid + j T, j < N; those from n on are the first one again
template <int N>
__device__ __forceinline__ bool vector_wait(gptr_word base, uint32_t n, uint32_t tag, uint32_t (&v)[N], const WalkBound &bound) {
    gptr_word at[N];
#pragma unroll
    for (int j = 0; j < N; j++) at[j] = base + (j * T + threadIdx.x < n ? j * T + threadIdx.x : 0);
    return words_wait<N>(at, tag, v, bound);
}

// the stream as the run before left it: x + y / rms(y) * weight
template <uint32_t KX>
__device__ __forceinline__ void settle(float (&x)[KX], const uint32_t (&y)[KX], const float (&yw)[KX], float n, float eps, float *red) {
    float sq = 0.0f;
#pragma unroll
    for (uint32_t j = 0; j < KX; j++) sq = __builtin_fmaf(__uint_as_float(y[j]), __uint_as_float(y[j]), sq);
    const float r = 1.0f / sqrtf(group_sum(sq, red) / n + eps);
#pragma unroll
    for (uint32_t j = 0; j < KX; j++) x[j] = __builtin_fmaf(__uint_as_float(y[j]) * r, yw[j], x[j]);
}
// its layer norm to LDS.  A wave's squares are taken from its own mean and moved to that of all: one exchange, no cancellation
template <typename El, uint32_t KX>
__device__ __forceinline__ void layer_norm(const float (&x)[KX], const float (&w)[KX], float eps, float2 *red, El *h) {
    constexpr float kOfWave = 64 * KX, kAll = kOfWave * kWaves;
    float sum = 0.0f, sq = 0.0f;
#pragma unroll
    for (uint32_t j = 0; j < KX; j++) sum += x[j];
    sum = wave_sum_f32(sum);
#pragma unroll
    for (uint32_t j = 0; j < KX; j++) {
        const float d = x[j] - sum / kOfWave;
        sq = __builtin_fmaf(d, d, sq);
    }
    sq = wave_sum_f32(sq);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = make_float2(sum, sq);
    __syncthreads();
    const float2 r = red[threadIdx.x & 15];
    const float mean = row_sum(r.x) / kAll, off = r.x / kOfWave - mean;
    const float scale = 1.0f / sqrtf(row_sum(__builtin_fmaf(kOfWave * off, off, r.y)) / kAll + eps);
#pragma unroll
    for (uint32_t j = 0; j < KX; j++) h[threadIdx.x + j * T] = from_f32<El>((x[j] - mean) * scale * w[j]);
}

// ---- the large products
template <typename El, uint32_t W>
__device__ __forceinline__ void vg_stream(const VgCtx &c, uint32_t idx, VgLds<El, W> &sm, u32x4 *staged) {
    using K = Vg<El, W>;
    constexpr uint32_t KX = K::KX, kPieceE = kPieceElems<El>;
    const RmiWalkVgArgs &a = c.a;
    const RmiWalkVgShape &s = a.s;
    uint32_t tid = threadIdx.x, wave = 0, lane = 0;
    El *h = reinterpret_cast<El *>(staged);
    u32x4 w[K::kHeld];
    // units: NP pieces a lane of a row each, B held; `base` of unit i
    auto load_unit = [&](uint32_t slot, gptr_u4 from) {
#pragma unroll
        for (uint32_t p = 0; p < K::NP; p++) w[slot * K::NP + p] = __builtin_nontemporal_load(from + p * 64 + lane);
    };
    auto first = [&](auto most, uint32_t n, auto base) {
#pragma unroll
        for (uint32_t i = 0; i < most.value && i < K::B; i++) {
            if (i < n) {
                load_unit(i, base(i));
            } else {  // (or what the phase before left would be kept)
#pragma unroll
                for (uint32_t p = 0; p < K::NP; p++) w[i * K::NP + p] = u32x4{0, 0, 0, 0};
            }
        }
    };
    auto product = [&](auto most, uint32_t n, auto base, auto operand, auto done) {
#pragma unroll
        for (uint32_t i = 0; i < most.value; i++) {
            if (i >= n) break;
            uint32_t at = lane;
            asm volatile("" : "+v"(at));  // (else the operand of all units is kept, which there is no room for)
            const u32x4 *hv = operand(i) + at;
            float acc = 0.0f;
#pragma unroll
            for (uint32_t p = 0; p < K::NP; p++) acc = dot_piece<El>(w[(i % K::B) * K::NP + p], hv[p * 64], acc);
            asm volatile("" : "+v"(acc));
            __builtin_amdgcn_sched_barrier(0);
            if (i + K::B < most.value && i + K::B < n) load_unit(i % K::B, base(i + K::B));
            done(i, wave_sum_f32(acc));
        }
    };
    auto vec = [&](const float *p, float (&v)[KX]) {
#pragma unroll
        for (uint32_t j = 0; j < KX; j++) v[j] = as_global<gptr_f32>(p)[tid + j * T];
    };
    using InUnits = std::integral_constant<uint32_t, K::kInUnits>;
    using Four = std::integral_constant<uint32_t, 4>;
    using Three = std::integral_constant<uint32_t, 3>;
    for (uint32_t run = 0; run < s.n_run; run++) {
        asm volatile("" : "+v"(tid));  // (what follows from it is worked out anew in every run, not kept and spilled)
        lane = tid & 63;
        wave = uint32_t(__builtin_amdgcn_readfirstlane(int(tid >> 6)));
        const uint32_t half = lane & 31, copy = lane >> 5;
        const uint32_t down0 = idx * K::kDownRows, down_n = down0 < W ? (W - down0 < K::kDownRows ? W - down0 : K::kDownRows) : 0;
        const RmiWalkVgRun::Stream y = table_entry(&a.runs[run].stream);
        const uint32_t tag = c.tag(run);
        const gptr_word from = c.from(run), to = c.to(run, copy);
        const uint32_t flags = uint32_t(__builtin_amdgcn_readfirstlane(int(y.flags)));  // (uniform: no value has to outlive the other branch)
        const bool delta = flags & RmiWalkVgRun::kDelta;
        const uint32_t rows = delta ? s.delta_rows : s.latent_rows, per = (rows + K::kStream - 1) / K::kStream;
        const uint32_t row0 = idx * per + wave, end = (idx + 1) * per < rows ? (idx + 1) * per : rows;
        const uint32_t n_in = row0 < end ? (end - row0 + kWaves - 1) / kWaves : 0;
        const uint32_t n_down = wave < down_n * 3 ? (down_n * 3 - wave + kWaves - 1) / kWaves : 0;
        auto down_base = [&](uint32_t i) {
            const uint32_t u = wave + i * kWaves;
            return as_global<gptr_u4>(y.w_down) + size_t(down0 + u / 3) * (s.ld_ff / kPieceE) + u % 3 * K::kRowPieces;
        };
        auto in_base = [&](uint32_t i) { return as_global<gptr_u4>(y.w_in) + size_t(row0 + i * kWaves) * (s.ld_w / kPieceE); };
        float x[KX], wn[KX], yw[KX];
        auto embedded = [&](const float *from, float (&v)[KX]) {  // by a launch in front, or here: without that launch a token is 14 us faster
            if (!a.embed.table) return vec(from, v);
#pragma unroll
            for (uint32_t j = 0; j < KX; j++) v[j] = embed_value<El>(a.embed, a.token, a.pos, tid + j * T);
        };
        // ---- the stream behind the run before
        auto stream_in = [&] {
            if (run == 0) {
                embedded(a.x, x);
                return;
            }
            uint32_t v[2 * KX], yv[KX];
            gptr_word p[2 * KX];
            const gptr_word before = c.from(run - 1);
#pragma unroll
            for (uint32_t j = 0; j < KX; j++) {
                p[j] = before + c.at.xb + tid + j * T;
                p[KX + j] = before + c.at.y + tid + j * T;
            }
            if (!words_wait<2 * KX>(p, tag - 1, v, c.bound)) sm.bad = 1;
#pragma unroll
            for (uint32_t j = 0; j < KX; j++) {
                x[j] = __uint_as_float(v[j]);
                yv[j] = v[KX + j];
            }
            settle<KX>(x, yv, yw, float(W), s.eps, sm.red[2]);
        };
        if (flags & RmiWalkVgRun::kLoopBegins) {
            const uint32_t n = wave < down_n * 2 ? (down_n * 2 - wave + kWaves - 1) / kWaves : 0;
            auto base = [&](uint32_t i) {
                const uint32_t u = wave + i * kWaves;
                return as_global<gptr_u4>(a.w_loop) + size_t(down0 + u / 2) * (s.ld_loop / kPieceE) + (u & 1) * K::kRowPieces;
            };
            float e[KX];
            if (run) vec(y.side_before, yw);
            embedded(a.embedded, e);
            first(Three{}, n, base);
            stream_in();
#pragma unroll
            for (uint32_t j = 0; j < KX; j++) {
                h[tid + j * T] = from_f32<El>(x[j]);
                h[W + tid + j * T] = from_f32<El>(e[j]);
            }
            __syncthreads();
            product(Three{}, n, base, [&](uint32_t i) { return staged + ((wave + i * kWaves) & 1) * K::kRowPieces; },
                    [&](uint32_t i, float z) { sm.s.part[wave + i * kWaves] = z; });
            __syncthreads();
            if (tid < 64 && half < down_n) word_store(to + c.at.xl + down0 + half, __float_as_uint(sm.s.part[2 * half] + sm.s.part[2 * half + 1]), tag);
            __syncthreads();
            vec(y.norm1, wn);
            first(InUnits{}, n_in, in_base);
            uint32_t v[KX];
            if (!vector_wait<KX>(from + c.at.xl, W, tag, v, c.bound)) sm.bad = 1;
#pragma unroll
            for (uint32_t j = 0; j < KX; j++) x[j] = __uint_as_float(v[j]);
        } else {
            vec(y.norm1, wn);
            if (run) vec(y.side_before, yw);
            first(InUnits{}, n_in, in_base);
            stream_in();
        }
        // ---- everything that reads it
        layer_norm<El, KX>(x, wn, s.eps, sm.stats, h);
        __syncthreads();
        {
            float mine = 0.0f;
            product(InUnits{}, n_in, in_base, [&](uint32_t) { return staged; }, [&](uint32_t i, float z) { mine = half == i ? z : mine; });
            const uint32_t row = row0 + half * kWaves;
            if (delta && row >= s.seg_g) mine *= sigmoid_t<El>(mine);
            if (half < n_in) word_store(to + c.at.in + row, __float_as_uint(mine), tag);
        }
        __syncthreads();  // (a late wave's words would wait behind the others' next weights)
        if (!delta) {  // ---- queries, keys and values from the latents
            const uint32_t q0 = idx * K::kUpQ + wave, q_end = (idx + 1) * K::kUpQ < kValues ? (idx + 1) * K::kUpQ : kValues;
            const uint32_t k0 = idx * K::kUpKv + wave, k_end = (idx + 1) * K::kUpKv < 2 * kValues ? (idx + 1) * K::kUpKv : 2 * kValues;
            const uint32_t q_pieces = s.q_rank / kPieceE, k_pieces = s.kv_rank / kPieceE;
#pragma unroll
            for (uint32_t i = 0; i < K::kUpQUnits; i++) {
                const uint32_t r = q0 + i * kWaves < q_end ? q0 + i * kWaves : 0;
#pragma unroll
                for (uint32_t p = 0; p < K::NPQ; p++)
                    w[i * K::NPQ + p] = __builtin_nontemporal_load(as_global<gptr_u4>(y.w_uq) + size_t(r) * (s.ld_q / kPieceE) + (p * 64 + lane < q_pieces ? p * 64 + lane : 0));
            }
#pragma unroll
            for (uint32_t i = 0; i < K::kUpKvUnits; i++) {
                const uint32_t r = k0 + i * kWaves < k_end ? k0 + i * kWaves : 0;
#pragma unroll
                for (uint32_t p = 0; p < K::NPK; p++)
                    w[K::kUpQUnits * K::NPQ + i * K::NPK + p] =
                        __builtin_nontemporal_load(as_global<gptr_u4>(y.w_ukv) + size_t(r) * (s.ld_kv / kPieceE) + (p * 64 + lane < k_pieces ? p * 64 + lane : 0));
            }
            // value i of both latents, one behind the other
            float l[2], ln[2], sq_q = 0.0f, sq_kv = 0.0f;
            uint32_t v[2];
            gptr_word p[2];
            const uint32_t all = s.q_rank + s.kv_rank;
#pragma unroll
            for (uint32_t j = 0; j < 2; j++) {
                const uint32_t i = tid + j * T < all ? tid + j * T : 0;
                p[j] = from + c.at.in + (i < s.q_rank ? i : s.seg_kv + i - s.q_rank);
                ln[j] = i < s.q_rank ? as_global<gptr_f32>(y.dq_norm)[i] : as_global<gptr_f32>(y.dkv_norm)[i - s.q_rank];
            }
            if (!words_wait<2>(p, tag, v, c.bound)) sm.bad = 1;
#pragma unroll
            for (uint32_t j = 0; j < 2; j++) {
                const uint32_t i = tid + j * T;
                l[j] = i < all ? __uint_as_float(v[j]) : 0.0f;
                sq_q = i < s.q_rank ? __builtin_fmaf(l[j], l[j], sq_q) : sq_q;
                sq_kv = i < s.q_rank ? sq_kv : __builtin_fmaf(l[j], l[j], sq_kv);
            }
            const float rq = 1.0f / sqrtf(group_sum(sq_q, sm.red[0]) / float(s.q_rank) + s.eps);
            const float rkv = 1.0f / sqrtf(group_sum(sq_kv, sm.red[1]) / float(s.kv_rank) + s.eps);
#pragma unroll
            for (uint32_t j = 0; j < 2; j++)
                if (tid + j * T < all) h[tid + j * T] = from_f32<El>(l[j] * (tid + j * T < s.q_rank ? rq : rkv) * ln[j]);
            __syncthreads();
            float mine = 0.0f;
            uint32_t row = 0;
            bool mine_is = false;
#pragma unroll
            for (uint32_t i = 0; i < K::kUpQUnits; i++) {
                float acc = 0.0f;
#pragma unroll
                for (uint32_t q = 0; q < K::NPQ; q++)
                    if (q * 64 + lane < q_pieces) acc = dot_piece<El>(w[i * K::NPQ + q], staged[q * 64 + lane], acc);
                acc = wave_sum_f32(acc);
                if (half == i) mine = acc, row = q0 + i * kWaves, mine_is = row < q_end;
            }
#pragma unroll
            for (uint32_t i = 0; i < K::kUpKvUnits; i++) {
                float acc = 0.0f;
#pragma unroll
                for (uint32_t q = 0; q < K::NPK; q++)
                    if (q * 64 + lane < k_pieces) acc = dot_piece<El>(w[K::kUpQUnits * K::NPQ + i * K::NPK + q], staged[q_pieces + q * 64 + lane], acc);
                acc = wave_sum_f32(acc);
                if (half == K::kUpQUnits + i) mine = acc, row = kValues + k0 + i * kWaves, mine_is = k0 + i * kWaves < k_end;
            }
            if (mine_is) word_store(to + c.at.up + row, __float_as_uint(mine), tag);
            __syncthreads();
        }
        // ---- the feed-forward
        {
            const uint32_t ff0 = (idx * kWaves + wave) * 4;
            auto base = [&](uint32_t i) { return as_global<gptr_u4>(y.w_ff) + size_t(ff0 + i) * (s.ld_w / kPieceE); };
            vec(y.norm2, wn);
            first(Four{}, 4, base);
            if (K::kDownAhead && n_down) {
#pragma unroll
                for (uint32_t p = 0; p < K::NP; p++)
                    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(down_base(0) + p * 64 + lane),
                                                     (__attribute__((address_space(3))) void *)&sm.s.down[wave * K::kRowPieces + p * 64], 16, 0, 2);
            }
            uint32_t v[KX];
            if (!vector_wait<KX>(from + c.at.xa, W, tag, v, c.bound)) sm.bad = 1;
#pragma unroll
            for (uint32_t j = 0; j < KX; j++) {
                x[j] = __uint_as_float(v[j]);
                const uint32_t i = tid + j * T - down0;  // (wraps below down0)
                if (i < down_n) sm.s.own[i] = x[j];
            }
            layer_norm<El, KX>(x, wn, s.eps, sm.stats, h);
            __syncthreads();
            float mine = 0.0f;
            product(Four{}, 4, base, [&](uint32_t) { return staged; }, [&](uint32_t i, float z) { mine = half == i ? z : mine; });
            const float o = fmaxf(mine, 0.0f) * dpp_f32<kDppQuadXor1>(mine);  // (gate, up) in lanes 2 i, 2 i + 1
            const uint32_t at = ff0 / 2;
            if constexpr (sizeof(El) == 2) {
                const float o1 = dpp_f32<kDppQuadXor2>(o);
                if (half == 0) word_store(to + c.at.ff + at / 2, uint32_t(f32_to_bf16(o)) | (uint32_t(f32_to_bf16(o1)) << 16), tag);
            } else {
                if (half == 0 || half == 2) word_store(to + c.at.ff + at + half / 2, __float_as_uint(o), tag);
            }
        }
        __syncthreads();
        {
            const float scale = as_global<gptr_f32>(y.ls2)[half < down_n ? down0 + half : 0];
#pragma unroll
            for (uint32_t i = 0; i < K::kDownHeld; i++)
                if (i + K::kDownAhead < n_down) load_unit(i, down_base(i + K::kDownAhead));
            constexpr uint32_t kWords = K::kFf * K::E / 4, N = (kWords + T - 1) / T;
            uint32_t v[N];
            if (!vector_wait<N>(from + c.at.ff, kWords, tag, v, c.bound)) sm.bad = 1;
#pragma unroll
            for (uint32_t j = 0; j < N; j++)
                if (j * T + tid < kWords) reinterpret_cast<uint32_t *>(staged)[j * T + tid] = v[j];
            __syncthreads();
#pragma unroll
            for (uint32_t i = 0; i < 3; i++) {
                if (i >= n_down) break;
                const uint32_t u = wave + i * kWaves;
                const u32x4 *hv = staged + u % 3 * K::kRowPieces + lane, *wv = sm.s.down + wave * K::kRowPieces + lane;
                float acc = 0.0f;
#pragma unroll
                for (uint32_t p = 0; p < K::NP; p++)
                    acc = dot_piece<El>(i < K::kDownAhead ? wv[p * 64] : w[(i - K::kDownAhead) * K::NP + p], hv[p * 64], acc);
                sm.s.part[u] = wave_sum_f32(acc);
            }
            __syncthreads();
            if (tid < 64 && half < down_n)
                word_store(to + c.at.xb + down0 + half,
                           __float_as_uint(__builtin_fmaf(scale, (sm.s.part[3 * half] + sm.s.part[3 * half + 1]) + sm.s.part[3 * half + 2], sm.s.own[half])), tag);
            __syncthreads();
        }
        if (sm.bad) break;
    }
}

// ---- a head of the delta rule
template <typename El, uint32_t W>
__device__ __forceinline__ void vg_delta(const VgCtx &c, uint32_t head, uint32_t run, VgLds<El, W> &sm) {
    const RmiWalkVgArgs &a = c.a;
    const RmiWalkVgShape &s = a.s;
    const RmiWalkVgRun::Delta y = table_entry(&a.runs[run].delta);
    auto &m = sm.c;
    uint32_t tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const uint32_t lane = tid & 63, group = kHeads / s.kv_heads, g = head / group, pos = a.pos;
    const uint32_t which = tid >> 7, ch = tid & (kDim - 1), channels = (2 * s.kv_heads + kHeads) * kDim;
    const uint32_t chan = (which == 0 ? g : which == 1 ? s.kv_heads + g : 2 * s.kv_heads + head) * kDim + ch;
    const bool has = which < 3, keeps = which == 2 || head % group == 0;
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
    const float rate = as_global<gptr_f32>(y.rate)[head], bias = as_global<gptr_f32>(y.bias)[head], norm = as_global<gptr_f32>(y.norm)[ch];
    constexpr uint32_t kSlices = T / 32, kPer = kDim / kSlices;
    const uint32_t quad = tid & 31, sl = tid >> 5;
    gptr_u4 st = as_global<gptr_u4>(a.now ? y.state[1] : y.state[0]) + size_t(head) * kDim * (kDim / 4) + quad;
    f32x4 r[kPer];
#pragma unroll
    for (uint32_t j = 0; j < kPer; j++) r[j] = __builtin_bit_cast(f32x4, st[size_t(sl * kPer + j) * (kDim / 4)]);
#pragma unroll
    for (uint32_t j = 0; j < kPer; j++) asm volatile("" ::"v"(r[j]));  // (before anything is stored)
    if (tid < 5 * kDim) {
        const uint32_t row = has ? chan : which == 3 ? s.seg_g + head * kDim + ch : (ch & 1 ? s.seg_a : s.seg_b) + head;
        const gptr_word at[1] = {c.from(run) + c.at.in + row};
        uint32_t v[1];
        if (!words_wait<1>(at, c.tag(run), v, c.bound)) sm.bad = 1;
        const float u = __uint_as_float(v[0]);
        if (has) {
            float z = 0.0f;
#pragma unroll
            for (uint32_t j = 0; j < 3; j++) z = __builtin_fmaf(taps[j], hist[j], z);
            z = __builtin_fmaf(taps[3], u, z);
            m.f[which][ch] = z * sigmoid_t<El>(z);
            if (keeps) {
                float *ho = a.now ? y.hist[0] : y.hist[1];
                const uint32_t off = 4 - s.taps;
#pragma unroll
                for (uint32_t j = 1; j < 3; j++)
                    if (j > off) ho[size_t(j - 1 - off) * channels + chan] = hist[j];
                ho[size_t(s.taps - 2) * channels + chan] = u;
            }
        } else if (which == 3) {
            m.f[3][ch] = u;
        } else if (ch < 2) {
            m.ba[ch] = ch ? expf(-rate * softplus_f32(u + bias)) : sigmoid_t<float>(u);
        }
    }
    __syncthreads();
    const float beta = m.ba[0], decay = m.ba[1];
    float qq = 0.0f, kk = 0.0f, kq = 0.0f;  // every wave for itself
#pragma unroll
    for (uint32_t d = 0; d < kDim; d += 64) {
        const float q = m.f[0][d + lane], k = m.f[1][d + lane];
        qq = __builtin_fmaf(q, q, qq);
        kk = __builtin_fmaf(k, k, kk);
        kq = __builtin_fmaf(k, q, kq);
    }
    const float rk = 1.0f / sqrtf(wave_sum_f32(kk) + 1e-6f), rq = 1.0f / sqrtf(wave_sum_f32(qq) + 1e-6f) / sqrtf(float(kDim));
    kq = wave_sum_f32(kq) * rk * rq;
    f32x4 pk = {0.f, 0.f, 0.f, 0.f}, pq = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (uint32_t j = 0; j < kPer; j++) {
        const float k = m.f[1][sl * kPer + j], q = m.f[0][sl * kPer + j];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            pk[e] = __builtin_fmaf(r[j][e], k, pk[e]);
            pq[e] = __builtin_fmaf(r[j][e], q, pq[e]);
        }
    }
    *reinterpret_cast<f32x4 *>(&m.part[0][sl][quad * 4]) = pk;
    *reinterpret_cast<f32x4 *>(&m.part[1][sl][quad * 4]) = pq;
    __syncthreads();
    if (tid < 2 * kDim) {
        float z = 0.0f;
#pragma unroll
        for (uint32_t i = 0; i < kSlices; i++) z += m.part[which][i][ch];
        m.sums[which][ch] = z;
    }
    __syncthreads();
    // (all waves: the values of channel ch)
    const float u = beta * (m.f[2][ch] - decay * (rk * m.sums[0][ch])), o = __builtin_fmaf(kq, u, decay * (rq * m.sums[1][ch]));
    const float sq = wave_sum_f32(o * o);
    if (tid < kDim) m.f[4][ch] = u;
    if (lane == 0) sm.red[3][tid >> 6] = sq;
    __syncthreads();
    const float scale = 1.0f / sqrtf((sm.red[3][0] + sm.red[3][1]) / float(kDim) + s.eps), out = o * scale * norm * m.f[3][ch];
    if (tid < 2 * kDim) {
        const uint32_t at = head * kDim + ch;
        if constexpr (sizeof(El) == 2) {
            const float other = dpp_f32<kDppQuadXor1>(out);
            if ((tid & 1) == 0) word_store(c.to(run, which) + c.at.act + at / 2, uint32_t(f32_to_bf16(out)) | (uint32_t(f32_to_bf16(other)) << 16), c.tag(run));
        } else {
            word_store(c.to(run, which) + c.at.act + at, __float_as_uint(out), c.tag(run));
        }
    }
    const f32x4 uq = *reinterpret_cast<const f32x4 *>(&m.f[4][quad * 4]);
    f32x4 *so = reinterpret_cast<f32x4 *>(a.now ? y.state[0] : y.state[1]) + size_t(head) * kDim * (kDim / 4) + quad;
#pragma unroll
    for (uint32_t j = 0; j < kPer; j++) {
        const float k = rk * m.f[1][sl * kPer + j];
        f32x4 n;
#pragma unroll
        for (int e = 0; e < 4; e++) n[e] = __builtin_fmaf(k, uq[e], decay * r[j][e]);
        so[size_t(sl * kPer + j) * (kDim / 4)] = n;
    }
}

// ---- every fourth block of a head's keys, and in part 0 the token's own: largest score, sum of the weights, weighted values
template <typename El, uint32_t W>
__device__ __forceinline__ void vg_attention(const VgCtx &c, uint32_t b, uint32_t run, VgLds<El, W> &sm) {
    const RmiWalkVgArgs &a = c.a;
    const RmiWalkVgShape &s = a.s;
    const RmiWalkVgRun::Latent y = table_entry(&a.runs[run].latent);
    auto &m = sm.c;
    uint32_t tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    constexpr uint32_t E = sizeof(El);
    const uint32_t head = b / kParts, part = b % kParts, lane = tid & 63, ch = tid & (kDim - 1), pos = a.pos;
    const uint32_t group = uint32_t(__builtin_amdgcn_readfirstlane(int(tid >> 7)));
    const uint32_t n_old = pos < s.window - 1 ? pos : s.window - 1, first = (pos - n_old) % s.capacity, off = first % kKeyBlock;
    const uint32_t n_blocks = (off + n_old + kKeyBlock - 1) / kKeyBlock, ring = s.capacity / kKeyBlock, first_block = first / kKeyBlock;
    // block j of this part: where it lies, and its first key's place among the keys (from n_old on and below zero: none)
    auto block_at = [&](uint32_t j) {
        const uint32_t bb = part + j * kParts;
        const uint32_t at = first_block + (bb < n_blocks ? bb : 0);
        return at < ring ? at : at - ring;  // (a ring's keys lie in one block more than it has, at most)
    };
    auto key_of = [&](uint32_t j) { return int((part + j * kParts) * kKeyBlock) - int(off); };
    constexpr uint32_t KP = kDim * E / 16, kPerRound = T / KP, kBpr = kPerRound / kKeyBlock, kRounds = (kPartBlocks + kBpr - 1) / kBpr;
    const uint32_t piece = tid % KP, krow = tid / KP;
    u32x4 kr[kRounds];
    gptr_u4 kc = as_global<gptr_u4>(y.k_cache) + size_t(head) * s.capacity * KP + piece;
#pragma unroll
    for (uint32_t i = 0; i < kRounds; i++) kr[i] = kc[size_t(block_at(i * kBpr + krow / kKeyBlock) * kKeyBlock + krow % kKeyBlock) * KP];
    constexpr uint32_t PB = kKeyBlock * E / 16, kGroups = T / kDim, kPerUnit = 16 / E;  // pieces of a block and channel, keys of one
    constexpr uint32_t kBpu = kGroups / PB, kUnits = (kPartBlocks + kBpu - 1) / kBpu;
    u32x4 vr[kUnits];
    gptr_u4 vc = as_global<gptr_u4>(y.v_cache) + size_t(head) * (s.capacity / kKeyBlock) * kDim * PB + ch * PB + group % PB;
#pragma unroll
    for (uint32_t i = 0; i < kUnits; i++) vr[i] = vc[size_t(block_at(i * kBpu + group / PB)) * kDim * PB];
    // which key of a block slot group % PB * kPerUnit + e holds
    auto slot_key = [&](uint32_t e) {
        const uint32_t sl = group % PB * kPerUnit + e;
        return E == 4 ? sl : (sl >> 3) * 4 + ((sl >> 2) & 1) * 16 + (sl & 3);
    };
#pragma unroll
    for (uint32_t i = 0; i < kUnits; i++) {  // values of no key, or of the token's own that another workgroup writes: zeros
        const int k0 = key_of(i * kBpu + group / PB);
        if (k0 >= 0 && k0 + int(kKeyBlock) <= int(n_old)) continue;
        u32x4 v = vr[i];
#pragma unroll
        for (uint32_t d = 0; d < 4; d++) {
            const uint32_t word = v[d];
            if constexpr (E == 4) {
                const int k = k0 + int(slot_key(d));
                v[d] = k >= 0 && k < int(n_old) ? word : 0u;
            } else {
                const int k = k0 + int(slot_key(2 * d));
                v[d] = (k >= 0 && k < int(n_old) ? word & 0xffffu : 0u) | (k + 1 >= 0 && k + 1 < int(n_old) ? word & 0xffff0000u : 0u);
            }
        }
        vr[i] = v;
    }
#pragma unroll
    for (uint32_t i = 0; i < kRounds; i++) asm volatile("" ::"v"(kr[i]));
#pragma unroll
    for (uint32_t i = 0; i < kUnits; i++) asm volatile("" ::"v"(vr[i]));
    // ---- the token's own
    if (tid < 3 * kDim) {
        const gptr_word at[1] = {c.from(run) + c.at.up + group * kValues + head * kDim + ch};
        uint32_t v[1];
        if (!words_wait<1>(at, c.tag(run), v, c.bound)) sm.bad = 1;
        const float u = __uint_as_float(v[0]);
        const uint32_t own = pos % s.capacity;
        if (group == 0) m.q[ch] = from_f32<El>(u);
        if (group == 1) {
            m.k[ch] = from_f32<El>(u);
            if (part == 0) static_cast<El *>(y.k_cache)[(size_t(head) * s.capacity + own) * kDim + ch] = from_f32<El>(u);
        }
        if (group == 2) {
            m.v[ch] = to_f32(from_f32<El>(u));
            const uint32_t k = own % kKeyBlock, slot = E == 4 ? k : ((k >> 2) & 3) * 8 + (k >> 4) * 4 + (k & 3);
            if (part == 0) static_cast<El *>(y.v_cache)[((size_t(head) * (s.capacity / kKeyBlock) + own / kKeyBlock) * kDim + ch) * kKeyBlock + slot] = from_f32<El>(u);
        }
    }
    __syncthreads();
    auto sum_key = [&](float v) {
        v += dpp_f32<kDppQuadXor1>(v);
        v += dpp_f32<kDppQuadXor2>(v);
        v += dpp_f32<kDppRowHalfMirror>(v);
        v += dpp_f32<kDppRowMirror>(v);
        return KP == 32 ? v + __shfl_xor(v, 16) : v;
    };
    const u32x4 q = reinterpret_cast<const u32x4 *>(m.q)[piece];
    float my_max = -INFINITY;
#pragma unroll
    for (uint32_t i = 0; i < kRounds; i++) {
        const uint32_t j = i * kBpr + krow / kKeyBlock;
        const int k = key_of(j) + int(krow % kKeyBlock);
        const bool live = j < kPartBlocks && k >= 0 && k < int(n_old);
        const float z = sum_key(dot_piece<El>(kr[i], q, 0.0f)) * s.attn_scale;
        if (j < kPartBlocks && piece == 0) m.p[j * kKeyBlock + krow % kKeyBlock] = live ? z : -INFINITY;
        my_max = live ? fmaxf(my_max, z) : my_max;
    }
    if (part == 0) {
        const float z = sum_key(dot_piece<El>(reinterpret_cast<const u32x4 *>(m.k)[piece], q, 0.0f)) * s.attn_scale;
        if (tid == 0) m.own_p = z;
        my_max = fmaxf(my_max, z);
    }
    my_max = fmaxf(my_max, __shfl_xor(my_max, 16));
    my_max = fmaxf(my_max, __shfl_xor(my_max, 32));
    if (lane == 0) sm.red[0][tid >> 6] = my_max;
    __syncthreads();
    float top = sm.red[0][0];
#pragma unroll
    for (uint32_t i = 1; i < kWaves; i++) top = fmaxf(top, sm.red[0][i]);
    float e = 0.0f;
    if (tid < kPartBlocks * kKeyBlock) {
        const int k = key_of(tid / kKeyBlock) + int(tid % kKeyBlock);
        const uint32_t r = tid % kKeyBlock, slot = E == 4 ? r : ((r >> 2) & 3) * 8 + (r >> 4) * 4 + (r & 3);
        if (k >= 0 && k < int(n_old)) e = exp_t<El>(m.p[tid] - top);
        m.weights[tid / kKeyBlock * kKeyBlock + slot] = from_f32<El>(e);
    } else if (tid < (kPartBlocks + 1) * kKeyBlock) {
        m.weights[tid] = from_f32<El>(0.0f);
    }
    if (tid == T - 1 && part == 0) {
        e = exp_t<El>(m.own_p - top);
        m.own_e = e;
    }
    const float total = group_sum(e, sm.red[1]);
    float acc = group == 0 && part == 0 ? m.v[ch] * to_f32(from_f32<El>(m.own_e)) : 0.0f;
#pragma unroll
    for (uint32_t i = 0; i < kUnits; i++)
        acc = dot_piece<El>(vr[i], reinterpret_cast<const u32x4 *>(m.weights)[(i * kBpu + group / PB) * PB + group % PB], acc);
    m.groups[group][ch] = acc;
    __syncthreads();
    if (tid < 2 * kDim) {
        const gptr_word to = c.to(run, group) + c.at.part + b * kPartWords;
        float o = 0.0f;
#pragma unroll
        for (uint32_t i = 0; i < kGroups; i++) o += m.groups[i][ch];
        word_store(to + ch, __float_as_uint(o), c.tag(run));
        if (ch < 2) word_store(to + kDim + ch, __float_as_uint(ch ? total : top), c.tag(run));
    }
}

// ---- a run's mixer, its output product, the token's gate and its projection
template <typename El, uint32_t W>
__device__ __forceinline__ void vg_chain(const VgCtx &c, uint32_t b, VgLds<El, W> &sm, u32x4 *staged) {
    using K = Vg<El, W>;
    constexpr uint32_t KX = K::KX, kPieceE = kPieceElems<El>;
    const RmiWalkVgArgs &a = c.a;
    const RmiWalkVgShape &s = a.s;
    auto &m = sm.c;
    El *h = reinterpret_cast<El *>(staged);
    const uint32_t own0 = b * K::kOwn;
    u32x4 wo[K::kOwnUnits][K::NPO];
    auto load_out = [&](const void *w, uint32_t t) {
        const uint32_t row0 = own0 + uint32_t(__builtin_amdgcn_readfirstlane(int(t >> 6))) * K::kOwnUnits;
#pragma unroll
        for (uint32_t i = 0; i < K::kOwnUnits; i++)
#pragma unroll
            for (uint32_t p = 0; p < K::NPO; p++)
                wo[i][p] = __builtin_nontemporal_load(as_global<gptr_u4>(w) + size_t(row0 + i) * (s.ld_v / kPieceE) + p * 64 + (t & 63));
    };
    const uint32_t token = a.embed.table ? a.token : a.tok[a.pos], id = token < s.vocab ? token : s.vocab - 1;
    for (uint32_t run = 0; run < s.n_run; run++) {
        const RmiWalkVgRun::Chain y = table_entry(&a.runs[run].chain);
        uint32_t tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const uint32_t lane = tid & 63, half = lane & 31, copy = lane >> 5, wave = uint32_t(__builtin_amdgcn_readfirstlane(int(tid >> 6)));
        const uint32_t tag = c.tag(run);
        const gptr_word from = c.from(run);
        const uint32_t flags = uint32_t(__builtin_amdgcn_readfirstlane(int(y.flags)));  // (uniform: no value has to outlive the other branch)
        const bool delta = flags & RmiWalkVgRun::kDelta;
        const float scale = as_global<gptr_f32>(y.ls1)[own0 + wave * K::kOwnUnits + (half < K::kOwnUnits ? half : 0)];
        // ---- own rows of the stream in front of the mixer
        if (run == 0 && !(flags & RmiWalkVgRun::kLoopBegins)) {
            if (tid < K::kOwn) m.own[tid] = a.embed.table ? embed_value<El>(a.embed, a.token, a.pos, own0 + tid) : a.x[own0 + tid];
        } else if (flags & RmiWalkVgRun::kLoopBegins) {
            if (tid < 64) {
                const gptr_word at[1] = {from + c.at.xl + own0 + (tid < K::kOwn ? tid : 0)};
                uint32_t v[1];
                if (!words_wait<1>(at, tag, v, c.bound)) sm.bad = 1;
                if (tid < K::kOwn) m.own[tid] = __uint_as_float(v[0]);
            }
        } else {
            uint32_t v[KX];
            float yw[KX], x[KX];
#pragma unroll
            for (uint32_t j = 0; j < KX; j++) {
                const uint32_t i = tid + j * T - own0;
                yw[j] = as_global<gptr_f32>(y.side_before)[tid + j * T];
                x[j] = i < K::kOwn ? m.own[i] : 0.0f;
            }
            if (!vector_wait<KX>(c.from(run - 1) + c.at.y, W, tag - 1, v, c.bound)) sm.bad = 1;
            settle<KX>(x, v, yw, float(W), s.eps, sm.red[2]);
#pragma unroll
            for (uint32_t j = 0; j < KX; j++) {
                const uint32_t i = tid + j * T - own0;
                if (i < K::kOwn) m.own[i] = x[j];
            }
        }
        __syncthreads();
        if (!delta)
            vg_attention<El, W>(c, b, run, sm);
        else if (b < kHeads)
            vg_delta<El, W>(c, b, run, sm);
        __syncthreads();
        if (!K::kOutAhead || run == 0) load_out(y.w_out, tid);
        // ---- the mixer's result
        if (delta) {
            constexpr uint32_t kWords = kValues * K::E / 4, N = kWords / T;
            uint32_t v[N];
            if (!vector_wait<N>(from + c.at.act, kWords, tag, v, c.bound)) sm.bad = 1;
#pragma unroll
            for (uint32_t j = 0; j < N; j++) reinterpret_cast<uint32_t *>(staged)[j * T + tid] = v[j];
        } else {
#pragma unroll 1
            for (uint32_t j = 0; j < kValues / T; j++) {  // (unrolled it would hold more than there is room for beside the weights)
                const gptr_word part = from + c.at.part + (wave * 64 + j * T) / kDim * kParts * kPartWords;  // this wave's head's
                gptr_word at[kParts + 1];
                uint32_t v[kParts + 1];
#pragma unroll
                for (uint32_t p = 0; p < kParts; p++) at[p] = part + p * kPartWords + tid % kDim;
                at[kParts] = part + (lane >> 1) % kParts * kPartWords + kDim + (lane & 1);
                if (!words_wait<kParts + 1>(at, tag, v, c.bound)) sm.bad = 1;
                float m[kParts], top = -INFINITY, total = 0.0f, o = 0.0f;
#pragma unroll
                for (uint32_t p = 0; p < kParts; p++) {
                    m[p] = __uint_as_float(uint32_t(__builtin_amdgcn_readlane(int(v[kParts]), int(p * 2))));
                    top = fmaxf(top, m[p]);
                }
#pragma unroll
                for (uint32_t p = 0; p < kParts; p++) {
                    const float f = exp_t<El>(m[p] - top);
                    o = __builtin_fmaf(f, __uint_as_float(v[p]), o);
                    total = __builtin_fmaf(f, __uint_as_float(uint32_t(__builtin_amdgcn_readlane(int(v[kParts]), int(p * 2 + 1)))), total);
                }
                h[tid + j * T] = from_f32<El>(o / total);
            }
        }
        __syncthreads();
        {
            float mine = 0.0f;
#pragma unroll
            for (uint32_t i = 0; i < K::kOwnUnits; i++) {
                float acc = 0.0f;
#pragma unroll
                for (uint32_t p = 0; p < K::NPO; p++) acc = dot_piece<El>(wo[i][p], staged[p * 64 + lane], acc);
                acc = wave_sum_f32(acc);
                mine = half == i ? acc : mine;
            }
            const uint32_t row = wave * K::kOwnUnits + half;
            if (half < K::kOwnUnits) word_store(c.to(run, copy) + c.at.xa + own0 + row, __float_as_uint(__builtin_fmaf(scale, mine, m.own[row])), tag);
        }
        __syncthreads();
        const uint32_t side_rows = s.side / kChain, side_pieces = s.side / kPieceE;
        const uint32_t g_row = tid / K::kRowPieces, g_at = tid % K::kRowPieces, p_row = tid / side_pieces, p_at = tid % side_pieces;
        const u32x4 wg = as_global<gptr_u4>(y.w_gate)[size_t(b * side_rows + (g_row < side_rows ? g_row : 0)) * (s.ld_w / kPieceE) + g_at];
        const u32x4 wp = as_global<gptr_u4>(y.w_proj)[size_t(own0 + (p_row < K::kOwn ? p_row : 0)) * (s.ld_side / kPieceE) + p_at];
        const float mul = to_f32(static_cast<const El *>(y.mul)[size_t(id) * s.mul_ld + b * side_rows + (half < side_rows ? half : 0)]);
        if (K::kOutAhead && run + 1 < s.n_run) load_out(table_entry(&a.runs[run + 1].chain).w_out, tid);
        // ---- the gate: the whole stream behind the feed-forward
        {
            uint32_t v[KX];
            if (!vector_wait<KX>(from + c.at.xb, W, tag, v, c.bound)) sm.bad = 1;
#pragma unroll
            for (uint32_t j = 0; j < KX; j++) {
                const uint32_t i = tid + j * T;
                h[i] = from_f32<El>(__uint_as_float(v[j]));
                if (i - own0 < K::kOwn) m.own[i - own0] = __uint_as_float(v[j]);
            }
            __syncthreads();
            const float z = wave_sum_f32(g_row < side_rows ? dot_piece<El>(wg, staged[g_at], 0.0f) : 0.0f);
            if (lane == 0) m.gate[wave] = z;
            __syncthreads();
            if (tid < 64 && half < side_rows) {
                float t = 0.0f;
#pragma unroll
                for (uint32_t i = 0; i < K::kRowPieces / 64; i++) t += m.gate[half * (K::kRowPieces / 64) + i];
                word_store(c.to(run, copy) + c.at.side + b * side_rows + half, __float_as_uint(apply_act<El>(kActGeluTanh, t, 0.0f, 0.0f) * mul), tag);
            }
        }
        // ---- its projection
        {
            if (tid < 128) {
                const gptr_word at[1] = {from + c.at.side + (tid < s.side ? tid : 0)};
                uint32_t v[1];
                if (!words_wait<1>(at, tag, v, c.bound)) sm.bad = 1;
                if (tid < s.side) h[tid] = from_f32<El>(__uint_as_float(v[0]));
            }
            __syncthreads();
            float z = p_row < K::kOwn ? dot_piece<El>(wp, staged[p_at], 0.0f) : 0.0f;
            z += dpp_f32<kDppQuadXor1>(z);
            z += dpp_f32<kDppQuadXor2>(z);
            z += dpp_f32<kDppRowHalfMirror>(z);
            if (side_pieces >= 16) z += dpp_f32<kDppRowMirror>(z);
            if (side_pieces >= 32) z += __shfl_xor(z, 16);
            const bool last = run + 1 == s.n_run;
            if (p_row < K::kOwn && p_at < 2) {
                if (!last) word_store(c.to(run, p_at) + c.at.y + own0 + p_row, __float_as_uint(z), tag);
                if (last && p_at == 0) a.y[own0 + p_row] = z;
            }
            if (last && tid < K::kOwn) a.x[own0 + tid] = m.own[tid];
            __syncthreads();
        }
        if (sm.bad) break;
    }
}

template <typename El, uint32_t W>
__global__ __launch_bounds__(T) void vogizen_walk_kernel(RmiWalkVgArgs a) {
    __shared__ VgLds<El, W> sm;
    __shared__ u32x4 staged[3 * W * sizeof(El) / 16];  // a product's operand
    const VgWords at = vg_words(a.s);
    gptr_word words = as_global<gptr_word>(a.words);
    const VgCtx c{a, at, words, words + die_half() * 2 * at.n, WalkBound{a.failed, a.spins}};
    if (threadIdx.x == 0) sm.bad = 0;
    if (a.embed.table && blockIdx.x == 0 && threadIdx.x == 0) *a.tok_out = a.token;
    __syncthreads();
    if (blockIdx.x < kChain)
        vg_chain<El, W>(c, blockIdx.x, sm, staged);
    else
        vg_stream<El, W>(c, blockIdx.x - kChain, sm, staged);
}

template <typename F>
auto with_kernel(const RmiWalkVgShape &s, F f) {
    if (s.elem_bytes == 2)
        return s.width == 1024 ? f(vogizen_walk_kernel<rmi_bf16, 1024>, Vg<rmi_bf16, 1024>{}) : f(vogizen_walk_kernel<rmi_bf16, 2048>, Vg<rmi_bf16, 2048>{});
    return s.width == 1024 ? f(vogizen_walk_kernel<float, 1024>, Vg<float, 1024>{}) : f(vogizen_walk_kernel<float, 2048>, Vg<float, 2048>{});
}

}  // namespace

bool rmi_walk_vogizen_fits(const RmiWalkVgShape &s) {
    if ((s.width != 1024 && s.width != 2048) || (s.side != 64 && s.side != 128) || s.taps < 2 || s.taps > 4 || s.kv_heads == 0 || kHeads % s.kv_heads) return false;
    return with_kernel(s, [&](auto kernel, auto k) {
        using K = decltype(k);
        auto in_fits = [](uint32_t rows) { return (rows + K::kStream - 1) / K::kStream <= kWaves * K::kInUnits; };
        if (!in_fits(s.delta_rows) || !in_fits(s.latent_rows) || s.q_rank > K::kMaxQ || s.kv_rank > K::kMaxKv) return false;
        int coop = 0, per_cu = 0;
        if (kChain + K::kStream > uint32_t(rmi_device_cus()) ||
            hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, rmi_device()) != hipSuccess || !coop ||
            hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, int(T), 0) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        return per_cu >= 1;
    });
}

size_t rmi_walk_vogizen_words(const RmiWalkVgShape &s) { return 4 * size_t(vg_words(s).n); }

int rmi_launch_walk_vogizen(const RmiWalkVgArgs &a, hipStream_t st) {
    const uint32_t keys = a.pos + 1 < a.s.window ? a.pos + 1 : a.s.window;
    if (a.pos == 0 || keys > kWalkVgKeys) return rmi_fail(RMI_HIP_E_INVALID, "position %u is not the walk's", a.pos);
    RmiWalkVgArgs copy = a;
    void *args[] = {&copy};
    return with_kernel(a.s, [&](auto kernel, auto k) -> int {
        RMI_HIP_CHECK(hipLaunchCooperativeKernel(reinterpret_cast<const void *>(kernel), dim3(kChain + decltype(k)::kStream), dim3(T), args, 0, st));
        return RMI_HIP_OK;
    });
}
