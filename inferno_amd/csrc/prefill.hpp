// Prefill (many tokens per expert): grouped dequant-GEMM on MFMA (prefill.hip).
#pragma once
#include "common.hpp"

namespace inferno {

// Weight kinds the MFMA GEMM dequantises (routed Q2_K/Q3_K/Q4_K, Q8_0 dense).
bool prefill_supported(int quant);
// True when the routed layer (gate/up kind, down kind, shapes) has the MFMA path.
bool prefill_routed_supported(int quant, int down_quant, size_t H, size_t I, size_t E);
// Assignments from which the routed layer takes the MFMA path (measured
// crossovers against the several-token decode kernels, with the shared
// expert of the MFMA path on the library GEMMs; INFERNO_PREFILL_MIN_ASSIGNMENTS
// overrides both). Without a shared expert (c1): 32 assignments 55.7 against
// 63.2 us on the decode kernels, 48 70.9 against 67.2, 64 82.5 against
// 71.5. With one (c2, c4): 48-56 decode (c2 T = 6 0.262 against 0.313 ms),
// 64 even (c2 T = 8 0.335 against 0.338), 70 and up MFMA (c4 T = 7 1.030
// against 1.015, T = 8 1.151 against 1.050, c2 T = 10 0.408 against 0.378).
constexpr size_t kPrefillMinAssignments = 48;
constexpr size_t kPrefillMinAssignmentsShared = 66;
// Several bf16 tokens below those counts, in a layer that the fused decode
// launches also take: the grouped GEMMs over scaled rows when the assignments'
// expert bytes outweigh their launches (nine against four, three of them short
// ones that the decode launches have no counterpart of; two more with a shared
// expert). Measured over 28 layers (H 1024 .. 6144, I 512 .. 2048, Q2_K / Q3_K /
// Q4_K, with and without a shared expert) of 2 to 8 tokens, decode / grouped in
// us: from 24 assignments and 130 MiB on at worst 1.5 % slower, 19 % faster on
// average (68 points; Q2_K H 6144 I 2048 24 assignments, 284 MiB 115 / 116,
// with a shared expert 32 of them 378 MiB 177 / 153; Q4_K H 2816 I 1280 24,
// 139 MiB 62 / 56; Q3_K H 4096 I 1536 40, 309 MiB 146 / 126), below it mostly
// slower (Q2_K H 4096 I 1536 20, 118 MiB 65 / 68; Q3_K H 2048 I 768 32, 62 MiB
// 50 / 53; Q4_K H 6144 I 512 24, 122 MiB 61 / 63; Q2_K H 6144 I 2048 16, 189
// MiB 85 / 92).
inline bool grouped_beats_decode(size_t A, size_t expert_bytes) {
  return A >= 24 && A * expert_bytes >= size_t(130) << 20;
}

// 32-bit words of the routed planner's scratch (tile lists and counts).
size_t prefill_plan_words(size_t A, size_t E);
// Halfs per row of the f16 activations the grouped GEMMs read (x16, h16): K
// values, the sums of every 16 of them in two f16 terms (K / 8 halfs: per 256
// values 16 first terms, then 16 second ones, in the k order of the values),
// and 128 bytes of padding: a tile reads the same 128 bytes of up to 128 rows
// at once, and rows of a multiple of 512 bytes apart put all of them on one
// or two of the 16 L2 channels.
HD constexpr size_t f16_pitch(size_t K) { return K + K / 8 + 64; }
// Where a row of K values holds term `term` (0 or 1) of the sum of its
// group-th 16 values.
HD constexpr size_t f16_sum_at(size_t K, size_t group, int term) {
  return K + 32 * (group / 16) + 16 * size_t(term) +
         ((group & 12) | ((group & 1) << 1) | ((group >> 1) & 1));
}
// The two terms of a group sum t: t / 16 (never past f16's range, as the
// values are not) rounded to f16, and the rest times 2^11.
__device__ __forceinline__ uint16_t f16_sum_term(float t, int term) {
  const float m = t * 0.0625f;
  const _Float16 hi = (_Float16)m;
  return __builtin_bit_cast(uint16_t, term == 0 ? hi : (_Float16)((m - (float)hi) * 2048.0f));
}

// Scaled rows (the grouped GEMMs of a few tokens): the same, with the values in
// units of a power of two per 256 of them, and behind the padding a fp32 per 32
// values, eight equal ones per unit, that brings sums back.
HD constexpr size_t f16_scale_at(size_t K) { return f16_pitch(K); }
HD constexpr size_t f16_scaled_pitch(size_t K) { return f16_pitch(K) + K / 16; }

// rows0 [n0, K0] and, unless n1 is 0, rows1 [n1, K1] (bf16 or fp32) as scaled
// rows, in one launch.
struct RowsToScale {
  const void* x;
  uint16_t* out;  // f16_scaled_pitch(K) apart, 8-byte aligned
  size_t rows, K;
};
int launch_scaled_rows(hipStream_t s, int x_dtype, const RowsToScale& r0, const RowsToScale& r1);

// x [rows, K] (bf16 or fp32) -> f16 rows of f16_pitch(K), round to nearest even.
int launch_to_f16(hipStream_t s, const void* x, int x_dtype, size_t rows, size_t K, uint16_t* out);

struct PrefillRouted {
  int quant, down_quant;
  const void *gate, *up, *down;  // packed experts [E][rows][blocks]
  const uint16_t* x16;           // [T] f16 rows of f16_pitch(H)
  const uint32_t* offsets;       // [E+1] from the dispatch
  const uint32_t* sorted;        // [A]
  const uint32_t* active;        // [E+1]
  const float* weights;          // [A] routing weights (folded into h)
  size_t T, k, E, H, I;
  uint16_t* h16;                 // [A] f16 rows of f16_pitch(I): SwiGLU intermediate
  float* y;                      // [A, H] per-assignment down rows
  uint32_t* plan;                // prefill_plan_words(A, E)
  // most rows one expert can take: T when every token's ids are distinct
  // (the layer's own top-k), 0 when unknown (caller ids: up to A)
  size_t max_rows;
  // a few tokens (prefill_few_takes): x16 and h16 are scaled rows, the gate/up
  // writes h32 [A, I] for launch_scaled_rows to turn into h16; else null
  float* h32;
};
// True when the scaled-row GEMMs take a layer: formats, widths and the
// alignment of the weights and of the rows.
bool prefill_few_takes(int quant, int down_quant, const void* gate, const void* up,
                       const void* down, const void* rows, size_t H, size_t I, size_t E);

// The tile lists of the layer inside p.plan, for the dispatch launch to fill
// (launch_dispatch with a plan) before launch_prefill_gate_up reads them.
PlanOut prefill_plan_out(const PrefillRouted& p);
// Routed gate/up (+SwiGLU, routing weight) over the dispatch groups: plans
// the expert tiles, then the GEMM; writes h16.
int launch_prefill_gate_up(hipStream_t s, const PrefillRouted& p);
// Routed down over the same tiles (after launch_prefill_gate_up): writes y.
int launch_prefill_down(hipStream_t s, const PrefillRouted& p);

// True when a dense (shared) expert of these formats and widths has the
// MFMA GEMMs (gate/up Q2_K/Q3_K/Q4_K/Q8_0, down also Q6_K).
bool prefill_dense_supported(int quant, int down_quant, size_t H, size_t Is);
// Dense expert over all T rows (gate/up format quant, down down_quant):
// h16 = silu(x G^T) * (x U^T); ys = h16 D^T.
// The Q8_0 shared expert of a batch of T tokens on library GEMMs (f16
// weights expanded per call, fp32 accumulation): taken by
// launch_prefill_dense when it is given a workspace of
// dense_blas_workspace_bytes and dense_blas_takes holds.
// dense_blas_fits: the shapes the path covers (the workspace is sized by it);
// dense_blas_takes: those, unless switched off.
bool dense_blas_fits(int quant, int down_quant, size_t T, size_t H, size_t Is);
bool dense_blas_takes(int quant, int down_quant, size_t T, size_t H, size_t Is);
size_t dense_blas_workspace_bytes(size_t T, size_t H, size_t Is);
int launch_dense_blas(hipStream_t s, const void* gate, const void* up, const void* down,
                      const uint16_t* x16, size_t T, size_t H, size_t Is, float* ys, void* ws,
                      void* lib_ws);
// The library's own workspace, shared by the calls of one stream.
size_t blas_lib_workspace_bytes();
// Router logits of T bf16 tokens as three bf16 library GEMMs over the exact
// three-term split of the fp32 router (fp32 accumulation): logits [T][E].
bool router_blas_fits(size_t T, size_t H, size_t E);
bool router_blas_takes(size_t T, size_t H, size_t E, int x_dtype);
size_t router_blas_workspace_bytes(size_t T, size_t H, size_t E);
int launch_router_blas(hipStream_t s, const uint16_t* x, const float* w, size_t T, size_t H,
                       size_t E, float* logits, void* terms_ws, void* lib_ws);
int launch_prefill_dense(hipStream_t s, int quant, int down_quant, const void* gate,
                         const void* up, const void* down, const uint16_t* x16, size_t T,
                         size_t H, size_t Is, uint16_t* h16, float* ys,
                         void* blas_ws = nullptr, void* lib_ws = nullptr);

// out = (residual + ys) + sum over ranks of y[t*k + r] (rank order); residual,
// ys may be null.
int launch_prefill_combine(hipStream_t s, const float* y, const float* ys, const float* residual,
                           size_t T, size_t k, size_t H, float* out);

}  // namespace inferno
