// What the universal product and its 32-bit matrix-core forms are launched with.
#pragma once
#include "common.h"

enum : int { EPI_STORE = 0, EPI_ADD = 1, EPI_SWIGLU = 2 };

struct GemmArgs {
    const void* A;
    const void* W;
    void* C;
    int M, N, K;
    int lda, ldw, ldc;
    // Grouped mode (group_offsets != null): group g's rows are list[group_offsets[g] .. group_offsets[g+1]).
    // A's row for list entry p is p / a_div, C's row is p.  Weights of group g start at W + g * w_group_stride elements.
    const int* group_offsets;
    const int* list;
    int a_div;
    long w_group_stride;
    int up_offset;  // EPI_SWIGLU: W row n is the gate row, W row n + up_offset the up row
    int act;        // EPI_STORE, EPI_ADD: an activation applied to the product (LLMX_ACT_*), with its parameters on the device
    const float* act_params;
    GluArgs glu;    // EPI_SWIGLU: the gated unit and its per-row values
};

// Whether the 32-bit matrix-core forms (gemm_f32_cores.hip) take this product of float32 operands into float32, and their launch:
// n_groups 0 for a dense product.
bool llmx_gemm_f32_cores_take(const GemmArgs& g, int n_groups);
int llmx_gemm_f32_cores(const GemmArgs& g, int epi, int n_groups, hipStream_t stream);
