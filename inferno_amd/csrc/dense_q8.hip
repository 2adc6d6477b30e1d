// Dense Q8_0 products over a batch of tokens: the shared expert by itself
// (inferno_q8_0_gate_up_swiglu, inferno_q8_0_matvec_add2) and inside a layer
// of a small batch (semantics: crates/backend/src/backend.rs:1578, :1682;
// block layout crates/gguf/src/lib.rs:1472-1499).
//
// Bound by the 34 bytes per 32 weights: 16 tokens need one 16x16x32 MFMA per
// 512 weights (544 bytes, ~190 cycles of one SIMD's share of HBM) and ~70
// cycles of VALU. What it takes is many short streams at once: a workgroup
// owns 16 weight rows (8 gate and 8 up rows, so that a 2048-wide gate/up is
// 256 workgroups), and its wavefronts split K by 256-value units, each with
// its own LDS region for the unit's weights and tokens, filled by the LDS DMA
// and moved to registers whole before the next unit's copies go out. No
// barrier until the sums of the wavefronts are added, in their order.
//
// Measured, H 6144 and Is 2048, bf16 tokens, both entry points together (stage,
// gate/up, stage, down), against the packed-f16 GEMVs they replace: 16 tokens
// 127 -> 26 us, 4 40 -> 28, 1 even, 128 938 -> 116, 512 3700 -> 435; error
// against fp64 of the gate/up 2.4e-7 -> 1.6e-7 (fp32 tokens 1.3e-6 -> 2.2e-7),
// of the down 2.2e-6 -> 1.3e-7. The scales cost 8 % of the gate/up at 512
// tokens (172 us without) and nothing of the down.
//
// The codes enter the MFMA as exact f16 integers, each 32-value block's sums
// are scaled by its d in fp32. Tokens are one f16 term (bf16 values, or the
// layer's f16 rows) or two (fp32 values: 22 bits), in units of a power of two
// that puts the largest value of each 32 (a weight block's own width) at 2^14
// .. 2^15: what f16 cannot hold of a value lies 2^-39 below the largest one of
// its block, whatever the rest of the row holds. A unit for the whole row
// instead loses a row beside one large value.
#include "dense_q8.hpp"

#include "scaled_rows.hpp"

namespace inferno {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kUnit = 256, kUnitBytes = 272, kPitch = 68;  // words per staged weight row
constexpr int kRows = 16;                                  // weight rows per workgroup
constexpr size_t kDenseQ8MaxTokens = size_t(1) << 19;      // grid height

using gptr_t = __attribute__((address_space(1))) const void*;
using lptr_t = __attribute__((address_space(3))) void*;
__device__ __forceinline__ void dma16(const uint8_t* base, uint32_t off, uint8_t* l) {
  __builtin_amdgcn_global_load_lds((gptr_t)(base + off), (lptr_t)l, 16, 0, 0);
}

// ------------------------------------------------------------------- staging

// A wavefront per 256 values of a row, four to a lane; eight lanes share the
// power of two of their 32 values.
template <typename XT, int TERMS>
__global__ void __launch_bounds__(256)
    stage_kernel(const XT* __restrict__ x, int K, uint16_t* __restrict__ staged) {
  const int lane = threadIdx.x & 63, kb = int(blockIdx.y) * 4 + int(threadIdx.x >> 6);
  if (kb * kUnit >= K) return;
  const int at = kb * kUnit + 4 * lane;
  uint16_t* out = staged + size_t(blockIdx.x) * dense_q8_pitch(K, TERMS);
  float v[4];
  scaled::load4(x + size_t(blockIdx.x) * K + at, v);
  const int e = scaled::run_exponent<32>(v);
  if ((lane & 7) == 0)
    reinterpret_cast<float*>(out + size_t(TERMS) * K)[kb * 8 + lane / 8] =
        __builtin_amdgcn_ldexpf(1.f, -e);
  _Float16 hi[4], lo[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float u = __builtin_amdgcn_ldexpf(v[j], e);
    hi[j] = (_Float16)u;
    lo[j] = (_Float16)(u - (float)hi[j]);
  }
  scaled::put4(out + at, hi);
  if constexpr (TERMS == 2) scaled::put4(out + K + at, lo);
}

// ---------------------------------------------------------------------- GEMM

__device__ __forceinline__ half2v as_h2(uint32_t v) { return __builtin_bit_cast(half2v, v); }

// Eight codes of two words (offset binary after the xor) as exact f16
// integers, order 0 2 1 3 4 6 5 7: 1024 + u under the exponent of 1024, minus
// 1152.
__device__ __forceinline__ half8 codes8(uint32_t w0, uint32_t w1) {
  const half2v m = {(_Float16)-1152.0f, (_Float16)-1152.0f};
  auto pair = [&](uint32_t w, uint32_t sel) {
    return __builtin_bit_cast(uint32_t, as_h2(__builtin_amdgcn_perm(0x64646464u, w, sel)) + m);
  };
  const uint32_t a = w0 ^ 0x80808080u, b = w1 ^ 0x80808080u;
  return __builtin_bit_cast(half8, make_uint4(pair(a, 0x04020400u), pair(a, 0x04030401u),
                                              pair(b, 0x04020400u), pair(b, 0x04030401u)));
}

// A wavefront's region: weights, tokens, the scales of 16 rows x 8 blocks.
template <int NB, int TERMS, int WAVES, bool SCALED>
constexpr size_t lds_bytes() {
  const size_t wave =
      kRows * kUnitBytes + size_t(NB) * TERMS * 16 * kUnit * 2 + (SCALED ? size_t(NB) * 512 : 0);
  return WAVES * wave;  // the sums passed between wavefronts take less
}

// NMAT = 2: gate rows n0 .. + 7 are the workgroup's rows 0 .. 7, up rows
// n0 .. + 7 its rows 8 .. 15; NMAT = 1: rows n0 .. + 15.
template <int NMAT, int NB, int TERMS, int WAVES, bool SCALED>
__global__ void __launch_bounds__(64 * WAVES) dense_q8_kernel(DenseQ8 p) {
  constexpr int TM = 16 * NB, TN = kRows / NMAT;
  constexpr int WBYTES = kRows * kUnitBytes, XBYTES = NB * TERMS * 16 * kUnit * 2;
  constexpr int SBYTES = SCALED ? NB * 512 : 0;
  static_assert(WAVES * NB * 4 * 64 * 4 <= int(lds_bytes<NB, TERMS, WAVES, SCALED>()), "sums fit");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem_d[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 15, g = lane >> 4;
  const int K = int(p.K), N = int(p.N), T = int(p.T);
  const int n0 = blockIdx.x * TN, t0 = blockIdx.y * TM;
  const int nkb = K / kUnit;
  const uint32_t row_bytes = uint32_t(nkb) * kUnitBytes;
  uint8_t* const wl = smem_d + wave * (WBYTES + XBYTES + SBYTES);
  uint8_t* const xl = wl + WBYTES;
  uint8_t* const sl = xl + XBYTES;

  // weight DMA: 17 lanes per row, three rows per instruction; rows past the
  // matrix are copies of its last one (not stored)
  const int lrow = lane / 17, piece = lane - 17 * lrow;
  constexpr int NI = (TN + 2) / 3;
  uint32_t woff[NI];
#pragma unroll
  for (int q = 0; q < NI; ++q)
    woff[q] = uint32_t(min(3 * q + lrow, N - 1 - n0)) * row_bytes + 16 * piece;
  const uint8_t* const w0 = static_cast<const uint8_t*>(p.w0) + size_t(n0) * row_bytes;
  const uint8_t* const w1 =
      NMAT == 2 ? static_cast<const uint8_t*>(p.w1) + size_t(n0) * row_bytes : nullptr;
  // token DMA: instruction u copies rows 2 u, 2 u + 1 of a term's 16-row
  // block, 32 pieces each, piece index xor'ed with the row
  const int xr = lane >> 5;
  const uint8_t* const xin = reinterpret_cast<const uint8_t*>(p.x + size_t(t0) * p.pitch);
  const uint32_t xpitch = uint32_t(p.pitch) * 2u;
  auto issue = [&](int kb) __attribute__((always_inline)) {
    const size_t wb = size_t(kb) * kUnitBytes;
#pragma unroll
    for (int m = 0; m < NMAT; ++m)
#pragma unroll
      for (int q = 0; q < NI; ++q)
        if (lrow < 3 && 3 * q + lrow < TN)
          dma16((m ? w1 : w0) + wb, woff[q], wl + (m * TN + 3 * q) * kUnitBytes);
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int t = 0; t < TERMS; ++t)
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int r = 16 * nb + 2 * u + xr;
          if (t0 + r < T)  // rows past the batch stay unwritten: their sums are not stored
            dma16(xin + size_t(kb) * 512 + size_t(t) * K * 2,
                  uint32_t(r) * xpitch + 16 * ((lane & 31) ^ (r & 15)),
                  xl + ((nb * TERMS + t) * 16 + 2 * u) * 512);
        }
    if constexpr (SCALED)  // the unit's eight scales of a row are two pieces
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
        if (lane < 32 && t0 + 16 * nb + (lane >> 1) < T)
          dma16(xin + p.scale_at * 2 + size_t(kb) * 32,
                uint32_t(16 * nb + (lane >> 1)) * xpitch + 16 * (lane & 1), sl + nb * 512);
  };

  floatx4 acc[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) acc[nb] = floatx4{0.f, 0.f, 0.f, 0.f};
  const uint32_t* const wr = reinterpret_cast<const uint32_t*>(wl) + i * kPitch;
  if (wave < nkb) issue(wave);
  for (int kb = wave; kb < nkb; kb += WAVES) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wavefront's own copies
    uint32_t ev[4][3], od[4][2], ds[4];
    half8 x[NB][TERMS][8];
    floatx4 sc[SCALED ? NB : 1][4][2];  // of token 4 g + v: blocks 0 .. 3, 4 .. 7
#pragma unroll
    for (int c = 0; c < 4; ++c) {  // blocks 2 c and 2 c + 1
#pragma unroll
      for (int j = 0; j < 3; ++j) ev[c][j] = wr[17 * c + 2 * g + j];
#pragma unroll
      for (int j = 0; j < 2; ++j) od[c][j] = wr[17 * c + 9 + 2 * g + j];
      ds[c] = (wr[17 * c] & 0xffffu) | (wr[17 * c + 8] & 0xffff0000u);
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int t = 0; t < TERMS; ++t)
#pragma unroll
        for (int k = 0; k < 8; ++k)
          x[nb][t][k] = *reinterpret_cast<const half8*>(xl + ((nb * TERMS + t) * 16 + i) * 512 +
                                                        16 * ((4 * k + g) ^ i));
    if constexpr (SCALED)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
          for (int j = 0; j < 2; ++j)
            sc[nb][v][j] = *reinterpret_cast<const floatx4*>(sl + (16 * nb + 4 * g + v) * 32 + 16 * j);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (kb + WAVES < nkb) issue(kb + WAVES);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int c = k >> 1;
      const half8 w = (k & 1) ? codes8(od[c][0], od[c][1])
                              : codes8(__builtin_amdgcn_alignbyte(ev[c][1], ev[c][0], 2),
                                       __builtin_amdgcn_alignbyte(ev[c][2], ev[c][1], 2));
      const float d = (float)as_h2(ds[c])[k & 1];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        floatx4 part = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = TERMS - 1; t >= 0; --t)
          part = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[nb][t][k], w, part, 0, 0, 0);
#pragma unroll
        for (int v = 0; v < 4; ++v)  // (the scale, a power of two, rounds nothing)
          acc[nb][v] += (SCALED ? part[v] * sc[nb][v][k >> 2][k & 3] : part[v]) * d;
      }
    }
  }

  // the wavefronts' sums in their order: wavefront nb adds those of token
  // block nb; sum v of lane (i, g) is token 4 g + v, row i
  __syncthreads();
  floatx4* const red = reinterpret_cast<floatx4*>(smem_d);  // [wave][nb][lane]
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) red[(wave * NB + nb) * 64 + lane] = acc[nb];
  __syncthreads();
  if (wave >= NB) return;
  floatx4 s = red[wave * 64 + lane];
#pragma unroll
  for (int w = 1; w < WAVES; ++w) s += red[(w * NB + wave) * 64 + lane];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int t = t0 + 16 * wave + 4 * g + v;
    const float y = s[v];
    if constexpr (NMAT == 2) {
      const float up = __shfl_xor(y, 8, 16);
      const int n = n0 + i;
      if (t < T && i < 8 && n < N) {
        const float h = silu(y) * up;
        if (p.out) p.out[size_t(t) * N + n] = h;
        if (p.h16)
          p.h16[size_t(t) * p.h_pitch + ((n & ~3) | ((n & 1) << 1) | ((n >> 1) & 1))] =
              __builtin_bit_cast(uint16_t, (_Float16)h);
      }
    } else {
      const int n = n0 + i;
      if (t < T && n < N) {
        const size_t o = size_t(t) * N + n;
        float r = p.res_a ? p.res_a[o] : 0.f;
        if (p.res_b) r += p.res_b[o];
        p.out[o] = r + y;
      }
    }
  }
}

template <int NMAT, int NB, int TERMS, int WAVES, bool SCALED>
int launch(hipStream_t s, const DenseQ8& p) {
  constexpr size_t lds = lds_bytes<NB, TERMS, WAVES, SCALED>();
  auto kern = dense_q8_kernel<NMAT, NB, TERMS, WAVES, SCALED>;
  if constexpr (lds > 64 * 1024) {
    static const hipError_t attr = hipFuncSetAttribute(
        reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
    INF_HIP(attr);
  }
  constexpr size_t TN = kRows / NMAT, TM = 16 * NB;
  const dim3 grid(unsigned((p.N + TN - 1) / TN), unsigned((p.T + TM - 1) / TM));
  kern<<<grid, 64 * WAVES, lds, s>>>(p);
  INF_LAUNCHED();
  return INFERNO_OK;
}

template <int NMAT, int NB, int TERMS, bool SCALED>
int launch_waves(hipStream_t s, const DenseQ8& p) {
  // few workgroups and a long K: as many wavefronts split it as LDS takes (up
  // to eight), so that a CU with one workgroup has more in flight
  constexpr int kMany = NB * TERMS == 1 ? 8 : 6;
  static_assert(lds_bytes<NB, TERMS, kMany, SCALED>() <= 160 * 1024, "LDS of a CU");
  const size_t wgs = (p.N * NMAT + kRows - 1) / kRows * ((p.T + 16 * NB - 1) / (16 * NB));
  if (wgs <= 384 && p.K / kUnit >= 16) return launch<NMAT, NB, TERMS, kMany, SCALED>(s, p);
  return launch<NMAT, NB, TERMS, 4, SCALED>(s, p);
}

// 32 tokens per workgroup only with one term (two would take 128 registers).
template <int NMAT>
int launch_terms(hipStream_t s, const DenseQ8& p) {
  if (p.terms == 2) return launch_waves<NMAT, 1, 2, true>(s, p);
  if (p.scale_at)
    return p.T > 16 ? launch_waves<NMAT, 2, 1, true>(s, p) : launch_waves<NMAT, 1, 1, true>(s, p);
  return p.T > 16 ? launch_waves<NMAT, 2, 1, false>(s, p) : launch_waves<NMAT, 1, 1, false>(s, p);
}

}  // namespace

bool dense_q8_takes(size_t T, const void* w0, const void* w1, const void* rows) {
  const uintptr_t a = reinterpret_cast<uintptr_t>(w0) | reinterpret_cast<uintptr_t>(w1) |
                      reinterpret_cast<uintptr_t>(rows);
  return T >= 1 && T <= kDenseQ8MaxTokens && a % 16 == 0;
}

int launch_dense_q8_stage(hipStream_t s, const void* x, int x_dtype, size_t T, size_t K,
                          uint16_t* staged) {
  const dim3 grid{unsigned(T), unsigned((K / kUnit + 3) / 4)};
  if (x_dtype == INFERNO_BF16)
    stage_kernel<uint16_t, 1><<<grid, 256, 0, s>>>(static_cast<const uint16_t*>(x), int(K), staged);
  else
    stage_kernel<float, 2><<<grid, 256, 0, s>>>(static_cast<const float*>(x), int(K), staged);
  INF_LAUNCHED();
  return INFERNO_OK;
}

int launch_dense_q8(hipStream_t s, const DenseQ8& p) {
  if (p.T == 0) return INFERNO_OK;
  if (p.K % kUnit || p.N == 0 || !(p.terms == 1 || (p.terms == 2 && p.scale_at))) {
    set_error("dense Q8_0 GEMM: K must be a multiple of 256, one term or two scaled ones");
    return INFERNO_ERR_INVALID;
  }
  return p.w1 ? launch_terms<2>(s, p) : launch_terms<1>(s, p);
}

}  // namespace inferno
