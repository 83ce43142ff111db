// The tiled GEMM over int8 weights (gemm_tile.hip), for llmserve_int8_linear_prefill.
#pragma once
#include "common.h"

namespace lsh {

int64_t int8_tile_workspace_bytes(int64_t M, int64_t N, int64_t K);
// K a multiple of 128; pointers 16-byte aligned; N K < 2^31.
void int8_tile_launch(const float* x, const int8_t* qweight, const float* scale, float* y, int64_t M, int64_t N,
                      int64_t K, void* workspace, hipStream_t st);

}  // namespace lsh
