// The float attention on the matrix instructions (attention_f32.hip), for the entry point that chooses between it and the
// kernel for any shape.
#pragma once

#include "common.h"
#include "score_shape.h"

namespace leone {

// part_acc (8 * rows * kv_heads * 16 * head_dim floats) and part_ml (8 * rows * kv_heads * 32), both or neither: a workgroup a share of a
// row's keys, merged by a second launch; the results are the same bits.
bool attention_f32_takes(const void* q, const void* out, const void* k_pool, const void* v_pool, int q_heads, int kv_heads, int head_dim,
                         int v_dim, int page_tokens);
void launch_attention_f32(const float* q, float* out, const float* k_pool, const float* v_pool, const int* positions, const int* row_entry,
                          const int* block_table, int max_blocks, int rows, int q_heads, int kv_heads, int head_dim, int page_tokens,
                          float scale, int window, const float* gate, long gate_stride, int keep_first, int gate_each,
                          const float* slopes, float temp_coef, int temp_every, const ScoreShape& shape, int chunk, float* part_acc,
                          float* part_ml, hipStream_t stream);

}  // namespace leone
