// A token of a Ruvenex session by one launch that walks all layers (walk_ruvenex.hip).
#ifndef RMI_WALK_RUVENEX_H
#define RMI_WALK_RUVENEX_H

#include "dense.h"
#include "seq_mixers.h"

struct RmiWalkRvLayer {  // in HBM, by role
    struct Attn {
        const float *conv, *cos_t, *sin_t;
        void *k_cache, *v_cache;
        float *hist[2];
    } attn;
    struct Recur {
        float *state[2];
        const float *norm;
    } recur;
    struct In {
        const void *w;
        const float *norm, *f_bias, *lower, *b1, *b2;
    } in;
    struct Out {
        const void *w;
    } out;
};

// Sizes that all layers share.
struct RmiWalkRvShape {
    uint32_t width, k_in, n_rows, in_ld, out_ld, k_attn, k_recur, k_pad;
    uint32_t seg[11];  // where the rows of q, k, v, gate, recurrence's q, f, v, the two gates and the feed-forward begin; their end
    uint32_t heads, kv_heads, recur_heads, taps, rot_dims, capacity, n_layer;
    float attn_scale, left_scale, right_scale, eps;
};

struct RmiWalkRvArgs {
    RmiWalkRvShape s;
    const RmiWalkRvLayer *layers;
    float *x;          // the token's embedding; left: the stream behind the last layer
    uint64_t *words;   // zeros at first
    uint32_t *failed;  // set where a wait did not end; the host's memory
    uint32_t tag0, spins, pos, now;
    RmiEmbed embed;    // with a table: the token is `token`, which the walk embeds itself and leaves in tok_out; else its embedding is in x
    uint32_t token;
    uint32_t *tok_out;
    const void *head;  // the vocabulary's rows, in_ld apart, or nullptr: no logits
    const float *head_norm;
    float *logits;
    uint32_t vocab;
    uint32_t n_output;  // workgroups of everything that ends in x
};

constexpr uint32_t kWalkRvMaxKeys = 512;  // of a head, in the registers of one workgroup
constexpr uint32_t kWalkRvSpins = 1u << 17;

bool rmi_walk_ruvenex_fits(const RmiWalkRvShape &s);
size_t rmi_walk_ruvenex_words(const RmiWalkRvShape &s);
// position a.pos, 1 .. kWalkRvMaxKeys - 1, bf16
int rmi_launch_walk_ruvenex(RmiWalkRvArgs a, hipStream_t st);

#endif  // RMI_WALK_RUVENEX_H
