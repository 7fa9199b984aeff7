// Generated tokens of a Qwen3 session by one launch that walks all layers, token after token (walk_qwen3.hip).
#ifndef RMI_WALK_QWEN3_H
#define RMI_WALK_QWEN3_H

#include "rmi_internal.h"

struct RmiWalkLayer {  // one layer's weights, in HBM
    const uint8_t *qkv, *o, *gu, *down;  // Q8_0 tile streams; q|k|v and gate|up stacked
    const float *attn_norm, *ffn_norm, *q_norm, *k_norm;  // the last two null if the model has none
};

struct RmiWalkShape {
    uint32_t n_embd, n_head, n_head_kv, head_dim_k, head_dim_v, n_ff, vocab, n_layer, kv_stride;
};

struct RmiWalkArgs {
    const RmiWalkLayer *layers;
    const uint8_t *embd, *head;
    const float *output_norm;
    const float *cos_t, *sin_t;    // [capacity][64]
    uint16_t *k_cache, *v_cache;   // [n_layer][capacity][kv_stride]
    float *x;                      // the embedding of the first step's token; left: that of the token behind the last step
    float *logits;                 // of the last step, where keep_logits
    uint64_t *words;               // the exchange between workgroups, zeros at first
    uint32_t *failed;              // set where a wait did not end
    uint32_t *tok, *step_argmax, *nonfinite;
    float *step_top2;
    void *sp;                      // StepParams
    uint32_t n_layer, n_head, n_head_kv, n_ff, vocab, capacity, kv_stride;
    uint32_t step0, n_steps, n_prompt;
    uint32_t tag0;                 // every word of this launch carries a tag above it
    uint32_t keep_logits;
    uint32_t n_attn, n_res, n_norm;  // workgroups by role (walk_roles)
    uint32_t spins;                  // how often a wait asks before it is given up
    float eps;
    int rounding;
};

// From this position on a head's keys are more than the walk holds.
constexpr uint32_t kWalkMaxKeys = 1280;
// Tokens of a launch, which holds every compute unit meanwhile.  us a token of 28 layers behind 100 keys with 1 | 2 | 4 | 8 | 16 of them 437 | 425 |
// 419 | 415 | 413; a product on host slices beside it, on another thread, 257 | 645 | 622 | 2264 | 5546 us, beside single launches 48.
constexpr uint32_t kWalkMaxSteps = 4;
constexpr uint32_t kWalkSpins = 1u << 17;  // at more than half a microsecond each

// Whether a session of this shape can be walked on this device.
bool rmi_walk_qwen3_fits(const RmiWalkShape &s);
size_t rmi_walk_qwen3_words(const RmiWalkShape &s);
// tags a launch of n_steps steps uses
inline uint32_t rmi_walk_qwen3_tags(uint32_t n_steps, uint32_t n_layer) { return n_steps * (n_layer + 1) + 1; }
// a.n_steps positions from a.step0 >= 1 on, all of them with fewer than kWalkMaxKeys keys
int rmi_launch_walk_qwen3(const RmiWalkShape &s, RmiWalkArgs a, hipStream_t st);

#endif  // RMI_WALK_QWEN3_H
