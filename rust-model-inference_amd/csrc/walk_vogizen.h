// A token of a Vogizen session by one launch that walks all layer runs (walk_vogizen.hip).
#ifndef RMI_WALK_VOGIZEN_H
#define RMI_WALK_VOGIZEN_H

#include "dense.h"
#include "seq_mixers.h"

struct RmiWalkVgRun {  // in HBM, by role; a layer as often as a token runs through it
    enum : uint64_t { kDelta = 1, kLoopBegins = 2 };
    struct Stream {
        const void *w_in, *w_ff, *w_down, *w_uq, *w_ukv;
        const float *norm1, *norm2, *ls2, *dq_norm, *dkv_norm;
        const float *side_before;  // the weight of what the run before leaves to be added
        uint64_t flags;
    } stream;
    struct Chain {
        const void *w_out, *w_gate, *w_proj, *mul;
        const float *ls1, *side_before;
        uint64_t flags;
    } chain;
    struct Delta {
        const float *conv, *rate, *bias, *norm;
        float *hist[2], *state[2];
    } delta;
    struct Latent {
        void *k_cache, *v_cache;
    } latent;
};

// Sizes that all runs share.
struct RmiWalkVgShape {
    uint32_t elem_bytes, width, n_run;
    uint32_t ld_w, ld_v, ld_ff, ld_q, ld_kv, ld_side, ld_loop;  // of rows of that many columns
    uint32_t side, mul_ld, vocab;
    uint32_t delta_rows, seg_b, seg_a, seg_g, kv_heads, taps;  // everything that reads the stream of a delta rule, and where its parts begin
    uint32_t latent_rows, q_rank, kv_rank, seg_kv, window, capacity;
    float attn_scale, eps;
};

struct RmiWalkVgArgs {
    RmiWalkVgShape s;
    const RmiWalkVgRun *runs;
    const void *w_loop;
    float *x;               // the token's embedding; left: the stream behind the last run, without
    float *y;               // what that run leaves to be added
    const float *embedded;  // the embedding, where there is a loop
    const uint32_t *tok;    // ids by position
    uint64_t *words;        // zeros at first
    uint32_t *failed;       // set where a wait did not end; the host's memory
    uint32_t tag0, spins, pos, now;
    RmiEmbed embed;    // with a table: the token is `token`, which the walk embeds itself and leaves in tok_out; else its embedding is in x
    uint32_t token;
    uint32_t *tok_out;
};

constexpr uint32_t kWalkVgKeys = 1024;  // most that a position sees, itself included
constexpr uint32_t kWalkVgSpins = 1u << 17;

bool rmi_walk_vogizen_fits(const RmiWalkVgShape &s);
size_t rmi_walk_vogizen_words(const RmiWalkVgShape &s);
// position a.pos, from 1 on, that sees at most kWalkVgKeys keys
int rmi_launch_walk_vogizen(const RmiWalkVgArgs &a, hipStream_t st);

#endif  // RMI_WALK_VOGIZEN_H
