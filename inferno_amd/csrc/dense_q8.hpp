// Dense Q8_0 expert (the shared expert) over a batch of tokens on the matrix
// cores (dense_q8.hip).
#pragma once
#include "common.hpp"

namespace inferno {

// Halfs per staged row of `terms` f16 terms of K values: the terms one after
// the other, a fp32 scale per 32 values, and padding off the L2 channel
// stride. Never more than the packed-f16 GEMV's staged row (gemv_stage_bytes)
// of the same row, which is what a caller's workspace holds: at K = 256, the
// narrowest, both take 640 (fp32 values 1152) bytes.
constexpr size_t dense_q8_pitch(size_t K, int terms) { return size_t(terms) * K + K / 16 + 48; }

// True when these kernels take a batch: T and the alignment of the weights
// (w1 null for one matrix) and of the staged rows.
bool dense_q8_takes(size_t T, const void* w0, const void* w1, const void* rows);

// Rows [T, K] as f16 terms (bf16 one, fp32 two), each 32 values in units of
// their own power of two: dense_q8_pitch rows.
int launch_dense_q8_stage(hipStream_t s, const void* x, int x_dtype, size_t T, size_t K,
                          uint16_t* staged);

struct DenseQ8 {
  const void *w0, *w1;    // gate and up, or one matrix and null: [N][K / 32] blocks
  const uint16_t* x;      // f16 rows (k order 0 2 1 3 4 6 5 7), `pitch` halfs apart
  size_t pitch;
  int terms;              // f16 terms per row
  size_t scale_at;        // a row's scales, one per 32 values: halfs from its start; 0: none
  size_t T, K, N;
  float* out;             // fp32 [T][N], or null
  uint16_t* h16;          // gate/up: f16 rows of h_pitch (the next GEMM's k order), or null
  size_t h_pitch;
  const float *res_a, *res_b;  // one matrix: added rows [T][N], or null
};
// two matrices: silu(x W0^T) * (x W1^T); one: res_a + res_b + x W0^T.
int launch_dense_q8(hipStream_t s, const DenseQ8& p);

}  // namespace inferno
