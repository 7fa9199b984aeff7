// Attention of a prompt pass, head dimension 128 (attn_prompt.hip).
#pragma once

#include "rmi_internal.h"

constexpr uint32_t kAttnPromptRows = 16;  // positions of a workgroup
// floats from one position's scores to the next: whole turns of 64 keys
inline uint32_t rmi_attn_prompt_score_stride(uint32_t n_keys) { return (n_keys + 63) / 64 * 64; }
// floats of scratch that hold at least one tile of sixteen positions of every head, and up to n_tok positions within 256 MB
inline size_t rmi_attn_prompt_scratch_floats(uint32_t n_head, uint32_t n_tok, uint32_t n_keys) {
    const size_t tile = size_t(n_head) * kAttnPromptRows * rmi_attn_prompt_score_stride(n_keys);
    const size_t tiles = (n_tok + kAttnPromptRows - 1) / kAttnPromptRows, most = (size_t(64) << 20) / tile;
    return tile * (tiles < most ? tiles : most > 1 ? most : 1);
}
// Positions step0 .. step0 + n_tok - 1, whose keys and values lie in the cache; q16 [n_tok][n_head][128], q8 likewise.
int rmi_launch_attn128_prompt(const uint16_t *q16, const uint16_t *k_cache, const uint16_t *v_cache, uint32_t step0, uint32_t n_tok,
                              uint32_t kv_stride, uint32_t n_head, uint32_t n_head_kv, float *scratch, size_t scratch_floats, int8_t *q8,
                              float *scales, int rounding, hipStream_t st);
