// Attention of a prompt pass, head dimension 128 (attn_prompt.hip).
#pragma once

#include "rmi_internal.h"

constexpr uint32_t kAttnPromptRows = 32;  // most positions of a workgroup
// floats from one position's scores to the next: whole turns of 128 keys
inline uint32_t rmi_attn_prompt_score_stride(uint32_t n_keys) { return (n_keys + 127) / 128 * 128; }
// floats of scratch that hold at least one tile of positions of every head, and up to n_tok positions within 256 MB
inline size_t rmi_attn_prompt_scratch_floats(uint32_t n_head, uint32_t n_tok, uint32_t n_keys) {
    const size_t tile = size_t(n_head) * kAttnPromptRows * rmi_attn_prompt_score_stride(n_keys);
    const size_t tiles = (n_tok + kAttnPromptRows - 1) / kAttnPromptRows, most = (size_t(64) << 20) / tile;
    return tile * (tiles < most ? tiles : most > 1 ? most : 1);
}
// Scratch for one layer's keys and values as limbs: blocks of 64 keys a head of either, and whether a block holds values
// that limbs don't.  blocks = 0: none, everything in f64.
struct RmiAttnLimbs {
    uint8_t *k = nullptr, *v = nullptr;
    uint32_t *wide = nullptr;
    uint32_t blocks = 0;
};
constexpr uint32_t kAttnLimbKeys = 32768;  // most keys whose weighted values' limbs add up in int32 (a session has 13 000 at most)
size_t rmi_attn_limbs_bytes(uint32_t n_head_kv, uint32_t capacity);
RmiAttnLimbs rmi_attn_limbs_at(void *base, uint32_t n_head_kv, uint32_t capacity);
// Whether a pass's attention is done in limbs, as far as its keys, values and queries let it.  limbs_hold: no query or key can
// be one that limbs don't hold, so far as the caller knows (a hint: the kernels look at all).
bool rmi_attn_prompt_in_limbs(uint32_t n_head, uint32_t step0, uint32_t n_tok, const RmiAttnLimbs &limbs, bool limbs_hold);
// Positions step0 .. step0 + n_tok - 1, whose keys and values lie in the cache; q16 [n_tok][n_head][128], q8 likewise.
int rmi_launch_attn128_prompt(const uint16_t *q16, const uint16_t *k_cache, const uint16_t *v_cache, uint32_t step0, uint32_t n_tok,
                              uint32_t kv_stride, uint32_t n_head, uint32_t n_head_kv, float *scratch, size_t scratch_floats,
                              const RmiAttnLimbs &limbs, bool limbs_hold, int8_t *q8, float *scales, int rounding, hipStream_t st);
