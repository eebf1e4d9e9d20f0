// What the universal attention and its float32 matrix-core form are launched with.
#pragma once
#include "common.h"

struct AttnArgs {
    const void* q;  // [T, n_heads * maps, head_dim]
    const void* k_cache;
    const void* v_cache;
    const int* pos;
    const int* row_entry;
    const int* tables;
    void* out;  // [T, n_heads * maps * v_dim]
    float scale;
    int n_heads, n_kv_heads, head_dim, page_tokens, max_blocks, window;
    int v_dim;   // width of a value head (the output's too); keys and queries have head_dim
    const float* gate;  // null, or float32 logits, row stride gate_ld: the output is multiplied by their sigmoid
    int gate_ld;
    int gate_wide;       // 0: a logit a (row, head); 1: a logit a (row, head, value dim)
    int keep_first, chunk, maps;
    float softcap;
    const float* slopes;   // [n_heads] or null
    const float* sink;     // [n_heads] or null
};

// Whether the float32 matrix-core form (attention_f32.hip) takes this attention (float32 in and out), and its launch; scratch (may be
// null): storage for the results of contexts that are shared out.
bool llmx_attention_f32_takes(const AttnArgs& a);
int llmx_attention_f32(const AttnArgs& a, int rows, float* scratch, long scratch_floats, hipStream_t stream);
