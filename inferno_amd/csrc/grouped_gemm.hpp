// Grouped dequant-GEMM on 16x16x32 f16 MFMA with every operand brought to LDS
// by the LDS DMA (global_load_lds): the expert GEMMs of prefill.hip over tiles
// of up to 64 rows.
//
// Work item: one tile of TM = 16 NB dispatch rows (tokens) of one expert x
// 16 RB weight rows per matrix and wavefront (four wavefronts). Lane (i =
// lane & 15, g = lane >> 4) of a wavefront dequantises, for each 32-value
// step, values 8 g .. 8 g + 7 of weight row i, which is how the K-quants lie
// in memory: 8 g indexes the 32-byte run whose bytes hold one value of each of
// the 2- or 4-bit planes, so a lane reads 8 bytes of quants per 128 (Q2_K,
// Q3_K) or 64 (Q4_K) values and uses every bit of them. The tokens are the A
// operand, the weights B: a lane's sums belong to its weight row.
//
// What bounds it, and the layout that follows. Few tokens per expert: the
// weights are read once, and HBM and the dequantisation take about the same
// time, so both have to run at once and each has to be cheap.
//  - Loads: no address arithmetic, register staging or LDS stores, only one
//    DMA instruction per 63 to 64 lanes. Each wavefront owns its rows: their
//    super-block lands in the wavefront's own LDS region and moves to
//    registers whole, and the DMA of the next super-block goes out into the
//    same region before the dequantisation starts. Few rows per workgroup (RB
//    = 1) and many workgroups per CU beat more rows (the partial 64-byte
//    sectors at a super-block's ends stay in L2 until the next step needs
//    them): 118 tiles of 3 rows, K = 6144, 2 x 2048 rows: Q2_K 0.251 ms
//    against 0.298 with RB = 2, Q3_K 0.357 against 0.433, Q4_K 0.340 against
//    0.376 (3.9, 3.6 and 4.9 TB/s); a second weight buffer per wavefront costs
//    more workgroups per CU than its prefetch gives (0.270, 0.373, 0.363).
//  - Dequantisation: see W<Q> (one packed multiply per two weights).
// Without the MFMAs and the dequantisation the same loads take 0.249, 0.287
// and 0.335 ms, without the loads the rest 0.189, 0.307 and 0.206: Q2_K and
// Q4_K are bound by their sectors, Q3_K by its dequantisation.
// Only the tokens are shared between wavefronts: one barrier per token buffer.
//
// Against the kernels of prefill.hip on these tiles (whole launches, gate/up
// and down): Q4_K, 16 tokens over 64 experts of 768 x 2048 39.9 + 22.1 -> 27.5
// + 16.3 us; Q3_K, 32 tokens over 128 experts of 1536 x 4096 252 + 131 -> 206
// + 107 us; Q3_K 64-row tiles of 2048 x 6144 experts 185 + 116 -> 180 + 92 us.
//
// Tokens lie in LDS without padding (the DMA writes 16 bytes per lane,
// contiguously); the 16-byte pieces of row i are stored exclusive-or'ed
// with i, so that the 16 rows of a fragment read touch all 64 banks.
#pragma once
#include <type_traits>

#include "gemv_common.hpp"
#include "prefill.hpp"

namespace inferno {
namespace grouped {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kUnit = 256;  // values per K unit (super-block / eight Q8_0 blocks)

struct GemmArgs {
  const uint8_t* w0;       // gate (or the down / single matrix)
  const uint8_t* w1;       // up, null for one matrix
  size_t stride;           // bytes per expert matrix
  const uint16_t* xin;     // f16 input rows (k order 0 2 1 3 4 6 5 7), f16_pitch(K) apart
  uint32_t in_div;         // input row = (sorted[c] or c) / in_div
  size_t in_rows;          // input rows
  const uint32_t* sorted;  // dispatch order, null = dense (identity)
  const float* route_w;    // routing weight per assignment, null = 1
  const uint4* tiles;      // {expert, c0, c1, 0}; null = dense tiles of TM rows
  const uint32_t* n_tiles;
  uint32_t rows;           // dense: number of rows
  int N, K;                // output rows per matrix, reduction length
  uint16_t* h_out;         // two matrices: f16 SwiGLU rows, f16_pitch(N) apart (k order as xin)
  float* h32;              // two matrices, scaled input rows: fp32 SwiGLU rows [*, N]
  float* y_out;            // one matrix: fp32 rows [*, N]
};

// This workgroup's expert and rows [c0, c1) of at most TM; false: none.
template <int TM>
__device__ __forceinline__ bool tile_of(const GemmArgs& p, uint32_t& e, uint32_t& c0,
                                        uint32_t& c1) {
  if (p.tiles == nullptr) {
    e = 0;
    c0 = blockIdx.y * TM;
    c1 = min(c0 + TM, p.rows);
  } else {
    if (blockIdx.y >= *p.n_tiles) return false;
    const uint4 tile = p.tiles[blockIdx.y];
    e = tile.x;
    c0 = tile.y;
    c1 = tile.z;
  }
  return c1 > c0;
}

__device__ __forceinline__ half2v as_h2(uint32_t v) { return __builtin_bit_cast(half2v, v); }
__device__ __forceinline__ uint32_t as_u32(half2v v) { return __builtin_bit_cast(uint32_t, v); }

// v(f) = f * mult + off for both f16 subnormal fields of a masked word, in f16.
__device__ __forceinline__ uint32_t fma_pair(uint32_t fields, float mult, float off) {
  const half2v f = as_h2(fields);
  const half2v r = {(_Float16)__builtin_fmaf((float)f[0], mult, off),
                    (_Float16)__builtin_fmaf((float)f[1], mult, off)};
  return as_u32(r);
}

// Eight values from bytes 0..7 of (w0, w1) with the field under `mask` (the
// same mask in both 16-bit halves, at bit position p): value = field * mult +
// off, mult already holding the 2^(24 - p). Output order 0 2 1 3 4 6 5 7.
__device__ __forceinline__ half8 dequant8(uint32_t w0, uint32_t w1, uint32_t mask, float mult,
                                          float off) {
  const uint32_t a = fma_pair(w0 & mask, mult, off);
  const uint32_t b = fma_pair((w0 >> 8) & mask, mult, off);
  const uint32_t c = fma_pair(w1 & mask, mult, off);
  const uint32_t d = fma_pair((w1 >> 8) & mask, mult, off);
  return __builtin_bit_cast(half8, make_uint4(a, b, c, d));
}

// f16 half `hi` of w, exactly widened, times m plus c in fp32 (v_fma_mix_f32).
__device__ __forceinline__ float mix_mul(uint32_t w, int hi, float m, float c) {
  const half2v h = as_h2(w);
  return __builtin_fmaf((float)h[hi], m, c);
}

__device__ __forceinline__ float ubyte_f32(uint32_t w, int b) {
  return float((w >> (8 * b)) & 0xffu);  // v_cvt_f32_ubyteN
}

// ---------------------------------------------------------- weight fragments
// W<Q>: half a super-block (128 values) of one row in registers. A row's
// super-block lies in LDS as kPitch words (DMA'd in kChunk-byte pieces,
// kLanes lanes per row); load<HALF>(row, g, odd) takes the words of the
// lane's 8-value group g, get<HALF, T>() returns the values 128 HALF + 32 T +
// 8 g .. + 7 (order 0 2 1 3 4 6 5 7). `odd`: the super-block starts 2 bytes
// into the first staged word (the 110- and 210-byte formats, of which whole
// words are staged).
//
// kExact: get() returns the integer (group scale) x (quant) times 2^-19,
// which f16 holds exactly, from two packed instructions per pair of values
// (mask in place, v_pk_mul_f16): the quant masked in place is the subnormal
// q 2^(p - 24), the group's multiplier is scale 2^(5 - p). The super-block
// factor d then scales the sums in fp32 (dscale()), once per super-block,
// and the offset terms enter as a product of their integers (offsets(), the
// sixteen groups of the super-block) with the group sums of the tokens.
// Forming the rounded value d sc q - dmin m per weight instead takes one
// v_fma_mixlo_f16 each, which issues at 8.6 cycles per wavefront against 5.2
// for a packed multiply of two (measured), and rounds every weight.

// Two integers 0 .. 63 under `mask` of w, as ((n - bias) * c0, (n - bias) * c1)
// in f16: 1024 + n under the exponent of 1024, then one exact fma.
__device__ __forceinline__ half2v int_pair(uint32_t w, uint32_t mask, float bias, float c0,
                                           float c1) {
  const half2v n = as_h2((w & mask) | 0x64006400u);
  const half2v c = {(_Float16)c0, (_Float16)c1};
  const half2v o = {(_Float16)(-(1024.0f + bias) * c0), (_Float16)(-(1024.0f + bias) * c1)};
  return __builtin_elementwise_fma(n, c, o);
}

// The four pairs (bytes 0 and 2, 1 and 3 of w0, then of w1) of masked fields
// times m.
__device__ __forceinline__ half8 scaled8(uint32_t w0, uint32_t w1, uint32_t mask, _Float16 m) {
  const half2v mm = {m, m};
  const uint32_t a = as_u32(as_h2(w0 & mask) * mm);
  const uint32_t b = as_u32(as_h2((w0 >> 8) & mask) * mm);
  const uint32_t c = as_u32(as_h2(w1 & mask) * mm);
  const uint32_t d = as_u32(as_h2((w1 >> 8) & mask) * mm);
  return __builtin_bit_cast(half8, make_uint4(a, b, c, d));
}

// The multiplier of step T: 2^(5 - bits), bits the position of its field.
constexpr float step_mult(int bits) {
  float v = 32.0f;
  for (int i = 0; i < bits; ++i) v *= 0.5f;
  return v;
}

template <int Q>
struct W;

// Q2_K [scales 16 | qs 64 | d | dmin]: value 128 h + 32 p + l uses
// q = (qs[32 h + l] >> 2 p) & 3 and scale byte 8 h + 2 p + l / 16: d sc q -
// dmin m (crates/gguf/src/lib.rs:1226-1293).
template <>
struct W<INFERNO_Q2_K> {
  static constexpr int kBytes = 84, kPitch = 21, kChunk = 4, kLanes = 21;
  static constexpr bool kHalfWord = false, kExact = true, kMin = true;
  uint32_t q[2];
  half2v s[2];
  template <int HALF>
  __device__ void load(const uint32_t* row, int g, uint32_t) {
    q[0] = row[4 + 8 * HALF + 2 * g];
    q[1] = row[5 + 8 * HALF + 2 * g];
    const int sh = 8 * (g >> 1);  // the lane's groups: bytes 0 and 2 after this shift
    s[0] = int_pair(row[2 * HALF] >> sh, 0x000f000fu, 0.f, step_mult(0), step_mult(2));
    s[1] = int_pair(row[2 * HALF + 1] >> sh, 0x000f000fu, 0.f, step_mult(4), step_mult(6));
  }
  template <int HALF, int T>
  __device__ half8 get() const {
    return scaled8(q[0], q[1], 0x00030003u << (2 * T), s[T >> 1][T & 1]);
  }
  // m of groups 8 (g & 1) .. + 7 as subnormals m 2^-24, times 2^11 for the
  // first terms of the group sums
  __device__ static half8 offsets(const uint32_t* row, int g, uint32_t) {
    const uint32_t a = row[2 * (g & 1)] >> 4, b = row[2 * (g & 1) + 1] >> 4;
    return scaled8(a, b, 0x000f000fu, (_Float16)(g < 2 ? 2048.f : 1.f));
  }
  __device__ static float dscale(const uint32_t* row, uint32_t) {
    return __builtin_amdgcn_ldexpf(f16_bits_to_f32_fast(uint16_t(row[20])), 19);
  }
  __device__ static float mscale(const uint32_t* row) {
    return __builtin_amdgcn_ldexpf(-f16_bits_to_f32_fast(uint16_t(row[20] >> 16)), 17);
  }
};

// Q3_K [hmask 32 | qs 64 | scales 12 | d]: value 128 n + 32 jj + l uses
// q = (qs[32 n + l] >> 2 jj) & 3, high bit hmask[l] bit (4 n + jj), 6-bit
// scale s6 of group 8 n + 2 jj + l / 16: d (s6 - 32) (q + 4 hbit - 4)
// (crates/gguf/src/lib.rs:1295-1367). get() gives (s6 - 32) u, u = q + 4
// hbit; the - 4 (s6 - 32) of every value is the offset term, in the same unit.
template <>
struct W<INFERNO_Q3_K> {
  static constexpr int kBytes = 110, kPitch = 28, kChunk = 4, kLanes = 28;
  static constexpr bool kHalfWord = true, kExact = true, kMin = false;
  uint32_t q[2], hm[2];
  half2v s[2];
  // the scale words (12 bytes) with their low bits at byte 0
  __device__ static void scale_words(const uint32_t* row, uint32_t sh, uint32_t o[3]) {
    const uint32_t a = row[24], b = row[25], c = row[26], d = row[27];
    o[0] = __builtin_amdgcn_alignbit(b, a, sh);
    o[1] = __builtin_amdgcn_alignbit(c, b, sh);
    o[2] = __builtin_amdgcn_alignbit(d, c, sh);
  }
  template <int HALF>
  __device__ void load(const uint32_t* row, int g, uint32_t odd) {
    const uint32_t sh = 16 * odd;
    uint32_t a[3], h[3], sw[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      a[j] = row[8 + 8 * HALF + 2 * g + j];
      h[j] = row[2 * g + j];
    }
    scale_words(row, sh, sw);
    q[0] = __builtin_amdgcn_alignbit(a[1], a[0], sh);
    q[1] = __builtin_amdgcn_alignbit(a[2], a[1], sh);
    hm[0] = __builtin_amdgcn_alignbit(h[1], h[0], sh);
    hm[1] = __builtin_amdgcn_alignbit(h[2], h[1], sh);
    const int gs = 8 * (g >> 1);  // the lane's groups: bytes 0 and 2 after this shift
    const uint32_t w0 = ((sw[0] >> (4 * HALF)) & 0x0f0f0f0fu) | (((sw[2] >> (4 * HALF)) & 0x03030303u) << 4);
    const uint32_t w1 = ((sw[1] >> (4 * HALF)) & 0x0f0f0f0fu) | (((sw[2] >> (4 * HALF + 2)) & 0x03030303u) << 4);
    s[0] = int_pair(w0 >> gs, 0x003f003fu, 32.f, step_mult(0), step_mult(2));
    s[1] = int_pair(w1 >> gs, 0x003f003fu, 32.f, step_mult(4), step_mult(6));
  }
  // u in place: q at bits 2 T, 2 T + 1 of the even (odd, shifted down) bytes,
  // hbit moved from bit 4 HALF + T to bit 2 T + 2
  template <int HALF, int T>
  __device__ half8 get() const {
    constexpr int up = 2 * T + 2 - (4 * HALF + T);
    constexpr uint32_t ql = 0x00030003u << (2 * T), hl = 0x00040004u << (2 * T);
    const half2v mm = {s[T >> 1][T & 1], s[T >> 1][T & 1]};
    auto field = [&](uint32_t qq, uint32_t h) {
      const uint32_t hs = up >= 0 ? h << (up >= 0 ? up : 0) : h >> (up < 0 ? -up : 0);
      return as_u32(as_h2((hs & hl) | (qq & ql)) * mm);
    };
    return __builtin_bit_cast(half8, make_uint4(field(q[0], hm[0]), field(q[0] >> 8, hm[0] >> 8),
                                                field(q[1], hm[1]), field(q[1] >> 8, hm[1] >> 8)));
  }
  // -4 (s6 - 32) 2^-19 of groups 8 (g & 1) .. + 7, times 16 for the first
  // terms of the group sums and 2^-7 for the second ones
  __device__ static half8 offsets(const uint32_t* row, int g, uint32_t odd) {
    uint32_t sw[3];
    scale_words(row, 16 * odd, sw);
    const int n = 4 * (g & 1);
    const uint32_t hi = sw[2] >> n;
    const uint32_t w0 = ((sw[0] >> n) & 0x0f0f0f0fu) | ((hi & 0x03030303u) << 4);
    const uint32_t w1 = ((sw[1] >> n) & 0x0f0f0f0fu) | (((hi >> 2) & 0x03030303u) << 4);
    const float c = g < 2 ? -0x1p-13f : -0x1p-24f;
    return __builtin_bit_cast(
        half8, make_uint4(as_u32(int_pair(w0, 0x003f003fu, 32.f, c, c)),
                          as_u32(int_pair(w0 >> 8, 0x003f003fu, 32.f, c, c)),
                          as_u32(int_pair(w1, 0x003f003fu, 32.f, c, c)),
                          as_u32(int_pair(w1 >> 8, 0x003f003fu, 32.f, c, c))));
  }
  __device__ static float dscale(const uint32_t* row, uint32_t odd) {
    return __builtin_amdgcn_ldexpf(f16_bits_to_f32_fast(uint16_t(row[27] >> (16 * odd))), 19);
  }
  __device__ static float mscale(const uint32_t*) { return 0.f; }
};

// Q4_K [d | dmin | scales 12 | qs 128]: value 64 c + 32 hh + l uses
// q = (qs[32 c + l] >> 4 hh) & 15 and the 6-bit (sc, m) of group 2 c + hh:
// d sc q - dmin m (crates/gguf/src/lib.rs:1369-1416). 144-byte rows are DMA'd
// 16 bytes per lane; 36 words apart, 16 rows start on 16 different multiples
// of 4 banks.
template <>
struct W<INFERNO_Q4_K> {
  static constexpr int kBytes = 144, kPitch = 36, kChunk = 16, kLanes = 9;
  static constexpr bool kHalfWord = false, kExact = true, kMin = true;
  uint32_t q[4];
  half2v s[2];
  template <int HALF>
  __device__ void load(const uint32_t* row, int g, uint32_t) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      q[2 * c] = row[4 + 16 * HALF + 8 * c + 2 * g];
      q[2 * c + 1] = row[5 + 16 * HALF + 8 * c + 2 * g];
    }
    uint32_t sc = row[1] & 0x3f3f3f3fu;
    if constexpr (HALF == 1) sc = (row[3] & 0x0f0f0f0fu) | ((row[1] >> 2) & 0x30303030u);
    // steps 0, 2 (low nibbles) and 1, 3
    s[0] = int_pair(sc, 0x00ff00ffu, 0.f, step_mult(0), step_mult(0));
    s[1] = int_pair(sc >> 8, 0x00ff00ffu, 0.f, step_mult(4), step_mult(4));
  }
  template <int HALF, int T>
  __device__ half8 get() const {
    return scaled8(q[2 * (T >> 1)], q[2 * (T >> 1) + 1], 0x000f000fu << (4 * (T & 1)),
                   s[T & 1][T >> 1]);
  }
  // m of the 32-value groups that hold 16-value groups 8 (g & 1) .. + 7, as
  // in Q2_K
  __device__ static half8 offsets(const uint32_t* row, int g, uint32_t) {
    const uint32_t lo = row[2] & 0x3f3f3f3fu;
    const uint32_t hi = ((row[3] >> 4) & 0x0f0f0f0fu) | ((row[2] >> 2) & 0x30303030u);
    const uint32_t m = (g & 1) ? hi : lo;
    const _Float16 c = (_Float16)(g < 2 ? 2048.f : 1.f);
    const half2v cc = {c, c};
    const uint32_t a = as_u32(as_h2(__builtin_amdgcn_perm(0u, m, 0x0c010c00u)) * cc);
    const uint32_t b = as_u32(as_h2(__builtin_amdgcn_perm(0u, m, 0x0c030c02u)) * cc);
    return __builtin_bit_cast(half8, make_uint4(a, a, b, b));
  }
  __device__ static float dscale(const uint32_t* row, uint32_t) {
    return __builtin_amdgcn_ldexpf(f16_bits_to_f32_fast(uint16_t(row[0])), 19);
  }
  __device__ static float mscale(const uint32_t* row) {
    return __builtin_amdgcn_ldexpf(-f16_bits_to_f32_fast(uint16_t(row[0] >> 16)), 17);
  }
};

// Q6_K [ql 128 | qh 64 | scales 16 (int8) | d]: value 128 h + 32 u + l uses
// q6 = (ql[64 h + 32 (u & 1) + l] >> 4 (u >> 1)) & 15 | ((qh[32 h + l] >> 2 u)
// & 3) << 4 and d sc[8 h + 2 u + l / 16] (q6 - 32)
// (crates/gguf/src/lib.rs:1418-1470). The 8-bit scale times the 6-bit quant
// does not fit f16's 11 bits: the value is formed in fp32 and rounded once.
template <>
struct W<INFERNO_Q6_K> {
  static constexpr int kBytes = 210, kPitch = 53, kChunk = 4, kLanes = 53;
  static constexpr bool kHalfWord = true, kExact = false, kMin = false;
  uint32_t ql[4], qh[2], sc[2];
  float d;
  template <int HALF>
  __device__ void load(const uint32_t* row, int g, uint32_t odd) {
    const uint32_t sh = 16 * odd;
    auto pair = [&](int w, uint32_t* o) {
      const uint32_t a = row[w], b = row[w + 1], c = row[w + 2];
      o[0] = __builtin_amdgcn_alignbit(b, a, sh);
      o[1] = __builtin_amdgcn_alignbit(c, b, sh);
    };
    pair(16 * HALF + 2 * g, ql);
    pair(16 * HALF + 8 + 2 * g, ql + 2);
    pair(32 + 8 * HALF + 2 * g, qh);
    const int gs = 8 * (g >> 1);
    const uint32_t s0 = row[48 + 2 * HALF], s1 = row[49 + 2 * HALF], s2 = row[50 + 2 * HALF];
    sc[0] = __builtin_amdgcn_alignbit(s1, s0, sh) >> gs;
    sc[1] = __builtin_amdgcn_alignbit(s2, s1, sh) >> gs;
    d = f16_bits_to_f32_fast(uint16_t(row[52] >> sh));
  }
  template <int HALF, int T>
  __device__ half8 get() const {
    auto six = [&](uint32_t w, uint32_t x) {
      return ((w >> (4 * (T >> 1))) & 0x0f0f0f0fu) | (((x >> (2 * T)) & 0x03030303u) << 4);
    };
    const uint32_t w0 = six(ql[2 * (T & 1)], qh[0]);
    const uint32_t w1 = six(ql[2 * (T & 1) + 1], qh[1]);
    const float dsc = d * float(int8_t((sc[T >> 1] >> (16 * (T & 1))) & 0xffu));
    return dequant8(w0, w1, 0x003f003fu, __builtin_amdgcn_ldexpf(dsc, 24), -32.0f * dsc);
  }
  // (named in code that kExact leaves out, never called)
  __device__ static half8 offsets(const uint32_t*, int, uint32_t) { return half8{}; }
  __device__ static float dscale(const uint32_t*, uint32_t) { return 1.f; }
  __device__ static float mscale(const uint32_t*) { return 0.f; }
};

// ------------------------------------------------------------------ kernel

using gptr_t = __attribute__((address_space(1))) const void*;
using lptr_t = __attribute__((address_space(3))) void*;

// Copies BYTES per lane from base + off (base the same in every lane) to l +
// BYTES * lane. The base stays opaque to the compiler, so that it is added in
// scalar registers and a lane keeps one 32-bit offset for all of its copies.
template <int BYTES>
__device__ __forceinline__ void dma(const uint8_t* base, uint32_t off, void* l) {
  const uint64_t v = reinterpret_cast<uint64_t>(base);
  uint64_t b = uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(v))))) |
               uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(v >> 32))))) << 32;
  asm("" : "+s"(b));
  const uint8_t* g = reinterpret_cast<const uint8_t*>(b) + off;
  if constexpr (BYTES == 16)
    __builtin_amdgcn_global_load_lds((gptr_t)g, (lptr_t)l, 16, 0, 0);
  else
    __builtin_amdgcn_global_load_lds((gptr_t)g, (lptr_t)l, 4, 0, 0);
}

constexpr int kWaves = 4;

// Halfs per token row of one LDS token buffer: a whole K unit for 16 tokens,
// half of one for 32, a 64-deep step above (two buffers of 128 tokens: 32 KB).
constexpr int x_halfs(int NB) { return NB == 1 ? 256 : NB == 2 ? 128 : 64; }

// [weights of the four wavefronts][two token buffers][two group-sum buffers]
// [two buffers of 16 scales]
template <int Q, int NMAT, int RB, int NB, bool SCALED>
constexpr size_t lds_bytes() {
  return size_t(kWaves) * NMAT * RB * 16 * W<Q>::kPitch * 4 + size_t(2) * 16 * NB * x_halfs(NB) * 2 +
         (W<Q>::kExact ? size_t(2) * NB * 1024 : 0) + (SCALED ? 128 : 0);
}

// Source of the weight DMA. A wavefront's instruction q copies rows [q RPI,
// + RPI) of its 16-row blocks, super-block kb: lane -> row lrow = lane /
// kLanes of them, piece lane % kLanes. The address is base (the same in every
// lane, from super-block 0 of row 0) plus a lane's offset, which is never
// negative. Half-word formats stage whole words: a super-block of odd index
// in its matrix (row * nkb + kb; rows start at multiples of 16) starts 2
// bytes into the word below it, one of even index ends 2 bytes before the end
// of its last word, which belongs to the next super-block (a matrix holds an
// even number of them). With an odd nkb (odd_rows) the two rows of one
// instruction differ in that: the base then lies 2 bytes low and the lanes of
// the even super-block add them back.
template <int Q>
struct WSrc {
  using F = W<Q>;
  static constexpr int RPI = 64 / F::kLanes;
  static_assert(!F::kHalfWord || RPI <= 2, "row parity of a lane");
  HD static int64_t base(int q, int kb, bool odd_rows, int64_t row_bytes) {
    int64_t b = int64_t(q * RPI) * row_bytes + int64_t(kb) * F::kBytes;
    if (F::kHalfWord) {
      if (!odd_rows) b -= 2 * (kb & 1);
      else if (RPI == 1) b -= 2 * ((kb + q) & 1);
      else b -= 2;
    }
    return b;
  }
  HD static uint32_t lane_off(int lane, int kb, bool odd_rows, uint32_t row_bytes) {
    const int lrow = lane / F::kLanes;
    uint32_t o = uint32_t(lrow) * row_bytes + uint32_t(F::kChunk * (lane - lrow * F::kLanes));
    if (F::kHalfWord && RPI == 2 && odd_rows) o += 2u * (1u - (uint32_t(kb + lrow) & 1u));
    return o;
  }
};

// One wavefront's DMA of its NMAT * 16 RB weight rows' super-block kb into its
// LDS region; off: WSrc::lane_off.
template <int Q, int NMAT, int RB>
__device__ __forceinline__ void issue_w(const uint8_t* s0, const uint8_t* s1, size_t row_bytes,
                                        uint32_t off, int kb, bool odd_rows, int lrow,
                                        uint8_t* dst) {
  using F = W<Q>;
  constexpr int RPI = WSrc<Q>::RPI;
  constexpr int RM = 16 * RB, NI = (RM + RPI - 1) / RPI;
#pragma unroll
  for (int m = 0; m < NMAT; ++m) {
#pragma unroll
    for (int q = 0; q < NI; ++q) {
      if (lrow < RPI && q * RPI + lrow < RM)
        dma<F::kChunk>((m ? s1 : s0) + WSrc<Q>::base(q, kb, odd_rows, int64_t(row_bytes)), off,
                       dst + (m * RM + q * RPI) * F::kPitch * 4);
    }
  }
}

// The lane's state that a K step needs.
template <int Q, int NMAT, int RB, int NB>
struct Lane {
  static constexpr int XH = x_halfs(NB), XP = XH / 8;
  static constexpr int XI = 16 * NB * XP / 64 / kWaves;  // token DMA instructions per wavefront
  const uint8_t *ws0, *ws1;  // weights: the wavefront's first rows
  size_t row_bytes;
  uint32_t woff[2];          // this lane's offset (WSrc::lane_off) for even and odd kb
  int lrow;
  bool odd_rows;
  const uint8_t* xin;        // tokens: all rows, and this lane's 16 bytes of buffer 0
  uint32_t xsrc[XI];
  bool xon[XI];
  uint32_t ssrc;             // group sums: this lane's 16 bytes of unit 0
  bool son;
  uint32_t csrc;             // scaled rows: this lane's scale of unit 0
  bool con;
  int xoff;                  // fragment read: byte offset in a token buffer
  int i, g;
};

// Token buffer SUB of K unit kb: the next buffer's DMA (with the next unit's
// group sums beside its first one), and after the unit's words are in
// registers its weights, go out; then the buffer's MFMAs run. The LDS written
// and the LDS read are different buffers, which the restrict qualifiers tell
// the compiler: it would otherwise wait for the copies before every fragment
// read.
template <int Q, int NMAT, int RB, int NB, bool SCALED, int SUB>
__device__ __forceinline__ void sub_step(const Lane<Q, NMAT, RB, NB>& L, const W<Q>* w, int kb,
                                         bool last, uint8_t* __restrict__ wdst,
                                         uint8_t* __restrict__ xdst, uint8_t* __restrict__ sdst,
                                         uint8_t* __restrict__ cdst,
                                         const uint8_t* __restrict__ xb, floatx4 (*acc)[NB]) {
  using LN = Lane<Q, NMAT, RB, NB>;
  constexpr int XH = LN::XH, SUBS = kUnit / XH, RT = NMAT * RB;
  constexpr bool kHalves = NB >= 4;  // w holds one half of the unit at a time
  if (SUB < SUBS - 1 || !last) {
    const size_t off = (size_t(kb) * SUBS + SUB + 1) * (XH * 2);
#pragma unroll
    for (int u = 0; u < LN::XI; ++u)
      if (L.xon[u]) dma<16>(L.xin + off, L.xsrc[u], xdst + u * 1024);
    if (W<Q>::kExact && SUB == SUBS - 1 && L.son) dma<16>(L.xin + size_t(kb + 1) * 64, L.ssrc, sdst);
    if (SCALED && L.con) dma<4>(L.xin + size_t(kb + 1) * 32, L.csrc, cdst);
  }
  if (SUB == (kHalves ? SUBS / 2 : 0) && !last) {
    // behind the tokens: the next buffer's wait leaves the weights in flight
    if constexpr (SUBS > 1) asm volatile("" ::: "memory");
    issue_w<Q, NMAT, RB>(L.ws0, L.ws1, L.row_bytes, (kb & 1) ? L.woff[0] : L.woff[1], kb + 1,
                         L.odd_rows, L.lrow, wdst);
  }
  auto step = [&](auto tc) __attribute__((always_inline)) {
    constexpr int KT = decltype(tc)::value;     // 32-value step within the buffer
    constexpr int ST = SUB * (XH / 32) + KT;    // within the unit
    // piece (4 KT + g) ^ swizzle(row): xoff holds the row base and 16 (g ^
    // swizzle); the step's bits of the index lie above the two of g
    const uint8_t* xr = xb + (L.xoff ^ (64 * KT));
    half8 b[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) b[nb] = *reinterpret_cast<const half8*>(xr + nb * 16 * XH * 2);
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const half8 a = w[kHalves ? r : 2 * r + ST / 4].template get<ST / 4, ST % 4>();
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
        acc[r][nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[nb], a, acc[r][nb], 0, 0, 0);
    }
  };
  step(std::integral_constant<int, 0>{});
  step(std::integral_constant<int, 1>{});
  if constexpr (XH >= 128) {
    step(std::integral_constant<int, 2>{});
    step(std::integral_constant<int, 3>{});
  }
  if constexpr (XH == 256) {
    step(std::integral_constant<int, 4>{});
    step(std::integral_constant<int, 5>{});
    step(std::integral_constant<int, 6>{});
    step(std::integral_constant<int, 7>{});
  }
}

// The sums of a tile to memory: sum v of lane (i, g) is token 4 g + v of its
// 16-token block, row i of its 16-row block.
template <int NMAT, int RB, int NB, bool SCALED>
__device__ __forceinline__ void store_tile(const GemmArgs& p, const floatx4 (*acc)[NB], uint32_t c0,
                                           uint32_t c1, int n0, int i, int g) {
  uint32_t asg[NB][4];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const uint32_t c = min(c0 + uint32_t(16 * nb + 4 * g + v), c1 - 1);
      asg[nb][v] = p.sorted ? p.sorted[c] : c;
    }
  float wts[NB][4];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int v = 0; v < 4; ++v)
      wts[nb][v] = (NMAT == 2 && p.route_w) ? p.route_w[asg[nb][v]] : 1.0f;
  // within four values the f16 rows hold 0 2 1 3
  const int ip = (i & ~3) | ((i & 1) << 1) | ((i >> 1) & 1);
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const bool on = c0 + uint32_t(16 * nb + 4 * g + v) < c1;
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        const int r0 = n0 + 16 * rb;
        if constexpr (NMAT == 2 && SCALED) {
          if (on)
            p.h32[size_t(asg[nb][v]) * p.N + r0 + i] =
                silu(acc[rb][nb][v]) * acc[RB + rb][nb][v] * wts[nb][v];
        } else if constexpr (NMAT == 2) {
          const _Float16 h = (_Float16)(silu(acc[rb][nb][v]) * acc[RB + rb][nb][v] * wts[nb][v]);
          uint16_t* row = p.h_out + size_t(asg[nb][v]) * f16_pitch(p.N);
          if (on) row[r0 + ip] = __builtin_bit_cast(uint16_t, h);
          // the sum of this group of 16 rows, in two f16 terms
          float t = (float)h;
#pragma unroll
          for (int o = 1; o < 16; o <<= 1) t += __shfl_xor(t, o, 16);
          if (on && i < 2) {
            row[f16_sum_at(p.N, r0 / 16, i)] = f16_sum_term(t, i);
          }
        } else {
          if (on) p.y_out[size_t(asg[nb][v]) * p.N + r0 + i] = acc[rb][nb][v];
        }
      }
    }
  }
}

// OCC: waves per SIMD the registers are budgeted for. SCALED: the input rows
// are f16_scaled_pitch apart, each 256 of their values in units of their own
// power of two, which the unit's sums are multiplied by (exactly); h stays
// fp32. For layers of a few tokens, whose other path (the decode launches)
// takes activations of any size: plain f16 rows lose h, which grows with the
// tokens' square, below 1e-3 and above 100 of a token's standard deviation.
// Four multiplications per 256 values and row block, under 1 % of the launch.
template <int Q, int NMAT, int RB, int NB, int OCC, bool SCALED = false>
__global__ void __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(OCC, 8)))
    wave_gemm_kernel(GemmArgs p) {
  using F = W<Q>;
  constexpr int TM = 16 * NB;
  constexpr int RM = 16 * RB;            // rows per matrix and wavefront
  constexpr int RT = NMAT * RB;          // 16-row blocks per wavefront
  constexpr int TN = kWaves * RM;        // rows per matrix and workgroup
  constexpr int XH = x_halfs(NB);        // halfs per token row of a buffer
  constexpr int XP = XH / 8;             // 16-byte pieces per token row
  constexpr int SUBS = kUnit / XH;       // token buffers per K unit
  constexpr int XROWS = 64 / XP;         // token rows per DMA instruction
  constexpr int XI = TM / XROWS / kWaves;  // DMA instructions per wavefront and buffer
  static_assert(XI >= 1 && XI * kWaves * XROWS == TM, "token rows split evenly");
  static_assert(NB <= kWaves, "one group-sum copy per wavefront");
  static_assert(!SCALED || (NB == 1 && F::kExact), "scales of one token block");
  constexpr int XBUF = TM * XH * 2;
  constexpr int WREG = RT * 16 * F::kPitch * 4;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem_g[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 15, g = lane >> 4;
  uint32_t e, c0, c1;
  if (!tile_of<TM>(p, e, c0, c1)) return;
  const int n0 = blockIdx.x * TN + wave * RM;  // this wavefront's first row
  const int K = p.K, nkb = K / kUnit;
  uint8_t* const wl = smem_g + wave * WREG;
  uint8_t* const xl = smem_g + kWaves * WREG;
  uint8_t* const sl = xl + 2 * XBUF;
  uint8_t* const cl = sl + 2 * NB * 1024;  // SCALED only
  const size_t pitch = SCALED ? f16_scaled_pitch(K) : f16_pitch(K);

  Lane<Q, NMAT, RB, NB> L;
  L.i = i;
  L.g = g;
  L.row_bytes = size_t(nkb) * F::kBytes;
  L.lrow = lane / F::kLanes;
  L.odd_rows = F::kHalfWord && (nkb & 1);
  const size_t wo = size_t(e) * p.stride + size_t(n0) * L.row_bytes;
#pragma unroll
  for (int b = 0; b < 2; ++b)
    L.woff[b] = WSrc<Q>::lane_off(lane, b, L.odd_rows, uint32_t(L.row_bytes));
  L.ws0 = p.w0 + wo;
  L.ws1 = NMAT == 2 ? p.w1 + wo : nullptr;
  // token DMA: instruction u of this wavefront fills buffer bytes
  // [(wave XI + u) 1024, + 1024): token row xr, piece (lane % XP) ^ swizzle.
  // Rows past the tile stay unwritten: their sums are not stored.
  auto swz = [](int row) { return XP >= 16 ? (row & 15) : ((row >> 1) & 7); };
  auto row_off = [&](int r) {
    const uint32_t cc = min(c0 + uint32_t(r), c1 - 1);
    const uint32_t a = p.sorted ? p.sorted[cc] : cc;
    return (a / p.in_div) * uint32_t(pitch) * 2u;
  };
#pragma unroll
  for (int u = 0; u < XI; ++u) {
    const int xr = (wave * XI + u) * XROWS + lane / XP;
    L.xon[u] = c0 + uint32_t(xr) < c1;
    L.xsrc[u] = row_off(xr) + 16 * ((lane % XP) ^ swz(xr));
  }
  // group sums: wavefront nb copies those of token block nb, 64 bytes a row
  L.son = wave < NB && c0 + uint32_t(16 * wave + (lane >> 2)) < c1;
  L.ssrc = row_off(16 * wave + (lane >> 2)) + uint32_t(K) * 2u + 16 * (lane & 3);
  // scales: wavefront 1 copies one of each row (a unit's eight are equal)
  L.con = SCALED && wave == 1 && lane < 16 && c0 + uint32_t(lane) < c1;
  L.csrc = SCALED ? row_off(lane & 15) + uint32_t(f16_scale_at(K)) * 2u : 0u;
  L.xin = reinterpret_cast<const uint8_t*>(p.xin);
  L.xoff = i * XH * 2 + 16 * (g ^ swz(i));

  floatx4 acc[RT][NB];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[r][nb] = floatx4{0.f, 0.f, 0.f, 0.f};

  uint8_t* const xw = xl + wave * XI * 1024;  // this wavefront's share of token buffer 0
  issue_w<Q, NMAT, RB>(L.ws0, L.ws1, L.row_bytes, L.woff[0], 0, L.odd_rows, L.lrow, wl);
#pragma unroll
  for (int u = 0; u < XI; ++u)
    if (L.xon[u]) dma<16>(L.xin, L.xsrc[u], xw + u * 1024);
  if (F::kExact && L.son) dma<16>(L.xin, L.ssrc, sl + wave * 1024);
  if (SCALED && L.con) dma<4>(L.xin, L.csrc, cl);
  constexpr int NW = NMAT * ((RM + WSrc<Q>::RPI - 1) / WSrc<Q>::RPI);  // weight DMAs per unit
  // up to 32 tokens: the whole super-block of every row in registers, the
  // region refilled at once; above, one half at a time beside the sums
  constexpr bool kHalves = NB >= 4;
  constexpr int WS = kHalves ? SUBS / 2 : 0;  // the sub-step that refills the weights
  W<Q> w[kHalves ? RT : 2 * RT];
  float ds[RT];
  floatx4 part[F::kExact ? RT : 1][NB];  // the unit's sums, in units of its d
  floatx4 offs[SCALED ? RT : 1], cs;     // SCALED: its offset terms, the tokens' scales
  const uint32_t* const wrd = reinterpret_cast<const uint32_t*>(wl) + i * F::kPitch;
  for (int kb = 0; kb < nkb; ++kb) {
    const bool last = kb + 1 == nkb;
    const uint32_t odd =
        F::kHalfWord ? (uint32_t(kb) + (L.odd_rows ? uint32_t(i) : 0u)) & 1u : 0u;
    // buffer of token sub-step S of this unit (SUBS is 1, 2 or 4)
    auto bufof = [&](int s) { return SUBS == 1 ? ((kb + s) & 1) : (s & 1); };
    auto sub = [&](auto sc) __attribute__((always_inline)) {
      constexpr int S = decltype(sc)::value;
      // this wavefront's share of the buffer (and, first in the unit, its
      // weights) has landed; after the barrier everyone's has, and the other
      // buffer is read by no one
      if (S == WS + 1 && !last)  // younger: the next unit's weights
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(NW) : "memory");
      else
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if constexpr (F::kExact && S == 0) {
        // the unit's offset terms: their integers times the group sums
        if constexpr (SCALED) cs = *reinterpret_cast<const floatx4*>(cl + (kb & 1) * 64 + g * 16);
        const uint8_t* sb = sl + (kb & 1) * (NB * 1024) + i * 64 + g * 16;
        half8 xs[NB];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) xs[nb] = *reinterpret_cast<const half8*>(sb + nb * 1024);
#pragma unroll
        for (int r = 0; r < RT; ++r) {
          const uint32_t* row = wrd + 16 * r * F::kPitch;
          const half8 o = F::offsets(row, g, odd);
          ds[r] = F::dscale(row, odd);
          const float ms = F::kMin ? F::mscale(row) : 0.f;
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) {
            const floatx4 m = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                xs[nb], o, floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
            if constexpr (F::kMin) {
              if constexpr (SCALED) offs[r] = m * ms;
              else acc[r][nb] += m * ms;
              part[r][nb] = floatx4{0.f, 0.f, 0.f, 0.f};
            } else {
              part[r][nb] = m;
            }
          }
          if constexpr (NB > 1) __builtin_amdgcn_sched_barrier(0);
        }
      }
      if constexpr (kHalves) {
        if constexpr (S == 0) {
#pragma unroll
          for (int r = 0; r < RT; ++r) w[r].template load<0>(wrd + 16 * r * F::kPitch, g, odd);
        }
        if constexpr (S == WS) {
#pragma unroll
          for (int r = 0; r < RT; ++r) w[r].template load<1>(wrd + 16 * r * F::kPitch, g, odd);
        }
      } else if constexpr (S == 0) {
#pragma unroll
        for (int r = 0; r < RT; ++r) {
          w[2 * r].template load<0>(wrd + 16 * r * F::kPitch, g, odd);
          w[2 * r + 1].template load<1>(wrd + 16 * r * F::kPitch, g, odd);
        }
      }
      // the words are in registers: the region is free for the next unit
      if constexpr (S == WS) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      sub_step<Q, NMAT, RB, NB, SCALED, S>(L, w, kb, last, wl, xw + (bufof(S) ^ 1) * XBUF,
                                   sl + ((kb & 1) ^ 1) * (NB * 1024) + wave * 1024,
                                   cl + ((kb & 1) ^ 1) * 64,
                                   xl + bufof(S) * XBUF, F::kExact ? part : acc);
    };
    sub(std::integral_constant<int, 0>{});
    if constexpr (SUBS >= 2) sub(std::integral_constant<int, 1>{});
    if constexpr (SUBS == 4) {
      sub(std::integral_constant<int, 2>{});
      sub(std::integral_constant<int, 3>{});
    }
    if constexpr (F::kExact) {
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          if constexpr (SCALED)
            acc[r][nb] += (F::kMin ? part[r][nb] * ds[r] + offs[r] : part[r][nb] * ds[r]) * cs;
          else
            acc[r][nb] += part[r][nb] * ds[r];
        }
    }
  }
  store_tile<NMAT, RB, NB, SCALED>(p, acc, c0, c1, n0, i, g);
}

}  // namespace grouped
}  // namespace inferno
