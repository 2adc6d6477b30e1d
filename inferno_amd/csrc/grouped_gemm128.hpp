// Grouped dequant-GEMM over tiles of up to 128 rows of one expert, on
// 32x32x16 f16 MFMA with LDS-DMA operands and exact integer weights
// (grouped_gemm.hpp has both).
//
// What bounds it: the matrix cores and the VALU at once. A fragment of 32
// weight rows x 16 values feeds four MFMAs of 32 cycles (128 tokens); each of
// them keeps the VALU's issue port for 8 cycles, the dequantisation takes 9
// to 17 packed instructions (~5 cycles each at two waves per SIMD), and what
// is left decides. So the sums stay where they are: instead of partial sums
// per super-block (128 more registers), the running sums are in units of the
// current super-block's d, and each new super-block first multiplies them by
// d_previous / d (64 multiplications per 16 fragments; the ratio's 2^-23 is
// far below the rounding of h). The group sums' products with the offsets
// (two MFMAs per sum, exact terms) go into the same sums: of formats with
// minima between two further multiplications, into units of dmin and back. A
// token fragment feeds two MFMAs (gate and up, or two blocks of down rows),
// which is half of what the LDS delivers.
//
// Two workgroups of four wavefronts per CU: weights of one super-block (each
// wavefront its own 64 rows, refilled when both halves are in registers), two
// 64-deep token buffers, the tokens' group sums.
//
// Measured, whole layers of 4096 tokens (H 6144, I 2048, 160 experts of which
// 8 per token, ~205 rows each) against f16-rounded weights from per-lane
// fragment loads or staged tiles: Q2_K 4.21 -> 3.89 ms, Q3_K 5.20 -> 4.35 ms,
// Q4_K 4.51 -> 4.15 ms; 2048 tokens Q3_K 3.10 -> 2.53 ms, error against fp64
// 4.3e-4 -> 3.4e-4 of the layer (what is left is h in f16).
#pragma once
#include "grouped_gemm.hpp"

namespace inferno {
namespace grouped {

typedef float floatx16 __attribute__((ext_vector_type(16)));

// T32<Q>: half a super-block (128 values) of one row for K steps of 16: lane
// (row i, kg = lane >> 5) takes values 16 S + 8 kg .. + 7 of step S (0 .. 7 of
// the half).
template <int Q>
struct T32;

template <>
struct T32<INFERNO_Q2_K> {
  uint32_t q[2][2];
  half2v s[4];  // [2 (S / 4) + S % 2][(S / 2) % 2]
  template <int HALF>
  __device__ void load(const uint32_t* row, int kg, uint32_t, bool live) {
#pragma unroll
    for (int par = 0; par < 2; ++par) {
      q[par][0] = row[4 + 8 * HALF + 4 * par + 2 * kg];
      q[par][1] = row[5 + 8 * HALF + 4 * par + 2 * kg];
    }
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      const uint32_t sc = live ? row[2 * HALF + w] : 0u;
      s[2 * w] = int_pair(sc, 0x000f000fu, 0.f, step_mult(4 * w), step_mult(4 * w + 2));
      s[2 * w + 1] = int_pair(sc >> 8, 0x000f000fu, 0.f, step_mult(4 * w), step_mult(4 * w + 2));
    }
  }
  template <int HALF, int S>
  __device__ half8 get() const {
    return scaled8(q[S & 1][0], q[S & 1][1], 0x00030003u << (2 * (S >> 1)),
                   s[2 * (S >> 2) + (S & 1)][(S >> 1) & 1]);
  }
};

template <>
struct T32<INFERNO_Q3_K> {
  uint32_t q[2][2], hm[2][2];
  half2v s[4];
  template <int HALF>
  __device__ void load(const uint32_t* row, int kg, uint32_t odd, bool live) {
    const uint32_t sh = 16 * odd;
#pragma unroll
    for (int par = 0; par < 2; ++par) {
      uint32_t a[3], h[3];
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        a[j] = row[8 + 8 * HALF + 4 * par + 2 * kg + j];
        h[j] = row[4 * par + 2 * kg + j];
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        q[par][j] = __builtin_amdgcn_alignbit(a[j + 1], a[j], sh);
        hm[par][j] = __builtin_amdgcn_alignbit(h[j + 1], h[j], sh);
      }
    }
    uint32_t sw[3];
    W<INFERNO_Q3_K>::scale_words(row, sh, sw);
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      const uint32_t s6 = ((sw[w] >> (4 * HALF)) & 0x0f0f0f0fu) |
                          (((sw[2] >> (4 * HALF + 2 * w)) & 0x03030303u) << 4);
      const uint32_t v = live ? s6 : 0x20202020u;  // scale 0
      s[2 * w] = int_pair(v, 0x003f003fu, 32.f, step_mult(4 * w), step_mult(4 * w + 2));
      s[2 * w + 1] = int_pair(v >> 8, 0x003f003fu, 32.f, step_mult(4 * w), step_mult(4 * w + 2));
    }
  }
  template <int HALF, int S>
  __device__ half8 get() const {
    constexpr int T = S >> 1, up = 2 * T + 2 - (4 * HALF + T);
    constexpr uint32_t ql = 0x00030003u << (2 * T), hl = 0x00040004u << (2 * T);
    const _Float16 m = s[2 * (S >> 2) + (S & 1)][T & 1];
    const half2v mm = {m, m};
    auto field = [&](uint32_t qq, uint32_t h) {
      const uint32_t hs = up >= 0 ? h << (up >= 0 ? up : 0) : h >> (up < 0 ? -up : 0);
      return as_u32(as_h2((hs & hl) | (qq & ql)) * mm);
    };
    const uint32_t* qq = q[S & 1];
    const uint32_t* h = hm[S & 1];
    return __builtin_bit_cast(half8, make_uint4(field(qq[0], h[0]), field(qq[0] >> 8, h[0] >> 8),
                                                field(qq[1], h[1]), field(qq[1] >> 8, h[1] >> 8)));
  }
};

template <>
struct T32<INFERNO_Q4_K> {
  uint32_t q[2][2][2];  // [chunk of 64][16-value half][word]
  half2v s[2];          // [low / high nibbles][chunk]
  template <int HALF>
  __device__ void load(const uint32_t* row, int kg, uint32_t, bool live) {
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int par = 0; par < 2; ++par) {
        q[c][par][0] = row[4 + 16 * HALF + 8 * c + 4 * par + 2 * kg];
        q[c][par][1] = row[5 + 16 * HALF + 8 * c + 4 * par + 2 * kg];
      }
    uint32_t sc = row[1] & 0x3f3f3f3fu;
    if constexpr (HALF == 1) sc = (row[3] & 0x0f0f0f0fu) | ((row[1] >> 2) & 0x30303030u);
    sc = live ? sc : 0u;
    s[0] = int_pair(sc, 0x00ff00ffu, 0.f, step_mult(0), step_mult(0));
    s[1] = int_pair(sc >> 8, 0x00ff00ffu, 0.f, step_mult(4), step_mult(4));
  }
  template <int HALF, int S>
  __device__ half8 get() const {
    constexpr int c = S >> 2, hh = (S >> 1) & 1;
    return scaled8(q[c][S & 1][0], q[c][S & 1][1], 0x000f000fu << (4 * hh), s[hh][c]);
  }
};

template <int Q, int NMAT>
constexpr size_t lds128_bytes() {
  return size_t(kWaves) * 64 * W<Q>::kPitch * 4 + 2 * 128 * 128 + 128 * 64;
}

// One 64-deep step: the copies it sends out, then four K steps.
template <int Q, int NMAT, int SUB>
__device__ __forceinline__ void sub128(const T32<Q>* w, const uint8_t* xbase, const uint32_t* xsrc,
                                       const bool* xon, bool xissue, uint8_t* __restrict__ xdst,
                                       const uint8_t* sbase, const uint32_t* ssrc,
                                       uint8_t* __restrict__ sdst, const uint8_t* ws0,
                                       const uint8_t* ws1, size_t row_bytes, uint32_t woff,
                                       int kbn, bool wissue, bool odd_rows, int lrow,
                                       uint8_t* __restrict__ wdst,
                                       const uint8_t* __restrict__ xb, int xoff,
                                       floatx16 (*acc)[4]) {
  constexpr int RB = NMAT == 2 ? 2 : 4;
  if (xissue) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (xon[u]) dma<16>(xbase, xsrc[u], xdst + u * 1024);
  }
  if constexpr (SUB == 2) {
    if (wissue) {
      asm volatile("" ::: "memory");  // behind the tokens: the next wait leaves these in flight
#pragma unroll
      for (int u = 0; u < 2; ++u) dma<16>(sbase, ssrc[u], sdst + u * 1024);
      issue_w<Q, NMAT, RB>(ws0, ws1, row_bytes, woff, kbn, odd_rows, lrow, wdst);
    }
  }
  auto step = [&](auto tc) __attribute__((always_inline)) {
    constexpr int KT = decltype(tc)::value, S = 4 * (SUB & 1) + KT;
    const uint8_t* xr = xb + (xoff ^ (32 * KT));
    half8 b[4];
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) b[nb] = *reinterpret_cast<const half8*>(xr + nb * 4096);
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const half8 a = w[r].template get<SUB / 2, S>();
#pragma unroll
      for (int nb = 0; nb < 4; ++nb)
        acc[r][nb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(b[nb], a, acc[r][nb], 0, 0, 0);
    }
  };
  step(std::integral_constant<int, 0>{});
  step(std::integral_constant<int, 1>{});
  step(std::integral_constant<int, 2>{});
  step(std::integral_constant<int, 3>{});
}

template <int Q, int NMAT>
__global__ void __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(2, 2)))
    tile128_gemm_kernel(GemmArgs p) {
  using F = W<Q>;
  constexpr int RB = NMAT == 2 ? 2 : 4, RM = 16 * RB, TN = kWaves * RM;
  constexpr int XBUF = 128 * 128;
  constexpr int WREG = 64 * F::kPitch * 4;
  constexpr int NW = NMAT * ((RM + WSrc<Q>::RPI - 1) / WSrc<Q>::RPI);  // weight DMAs per unit
  static_assert(NW + 2 < 64, "copies in flight fit the counter");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem_g[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 31, kg = lane >> 5;
  uint32_t e, c0, c1;
  if (!tile_of<128>(p, e, c0, c1)) return;
  const int n0 = blockIdx.x * TN + wave * RM;  // this wavefront's first row
  const int K = p.K, nkb = K / kUnit;
  uint8_t* const wl = smem_g + wave * WREG;
  uint8_t* const xl = smem_g + kWaves * WREG;
  uint8_t* const sl = xl + 2 * XBUF;
  uint8_t* const xw = xl + wave * 4096;  // this wavefront's share of token buffer 0
  uint8_t* const sw = sl + wave * 2048;

  const size_t row_bytes = size_t(nkb) * F::kBytes;
  const int lrow = lane / F::kLanes;
  const bool odd_rows = F::kHalfWord && (nkb & 1);
  const size_t wo = size_t(e) * p.stride + size_t(n0) * row_bytes;
  const uint8_t* const ws0 = p.w0 + wo;
  const uint8_t* const ws1 = NMAT == 2 ? p.w1 + wo : nullptr;
  const uint32_t woff0 = WSrc<Q>::lane_off(lane, 0, odd_rows, uint32_t(row_bytes));
  const uint32_t woff1 = WSrc<Q>::lane_off(lane, 1, odd_rows, uint32_t(row_bytes));
  const uint8_t* const xin = reinterpret_cast<const uint8_t*>(p.xin);
  auto row_off = [&](int r) {
    const uint32_t cc = min(c0 + uint32_t(r), c1 - 1);
    const uint32_t a = p.sorted ? p.sorted[cc] : cc;
    return (a / p.in_div) * uint32_t(f16_pitch(K)) * 2u;
  };
  // tokens: instruction u of this wavefront copies eight rows, eight pieces
  // each, piece index xor'ed with the row pair; rows past the tile stay
  // unwritten (their sums are not stored). Group sums: 16 rows of 64 bytes.
  uint32_t xsrc[4], ssrc[2];
  bool xon[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int xr = 32 * wave + 8 * u + (lane >> 3);
    xon[u] = c0 + uint32_t(xr) < c1;
    xsrc[u] = row_off(xr) + 16 * ((lane & 7) ^ ((xr >> 1) & 7));
  }
#pragma unroll
  for (int u = 0; u < 2; ++u)
    ssrc[u] = row_off(32 * wave + 16 * u + (lane >> 2)) + uint32_t(K) * 2u + 16 * (lane & 3);
  const int xoff = i * 128 + 16 * (kg ^ ((i >> 1) & 7));

  floatx16 acc[2][4];
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[r][nb][v] = 0.f;
  float unit[2] = {0.f, 0.f};  // the d that the sums are in units of (0: none yet)

  issue_w<Q, NMAT, RB>(ws0, ws1, row_bytes, woff0, 0, odd_rows, lrow, wl);
#pragma unroll
  for (int u = 0; u < 2; ++u) dma<16>(xin, ssrc[u], sw + u * 1024);
#pragma unroll
  for (int u = 0; u < 4; ++u)
    if (xon[u]) dma<16>(xin, xsrc[u], xw + u * 1024);

  T32<Q> w[2];
  bool live[2];
  const uint32_t* const wrd = reinterpret_cast<const uint32_t*>(wl) + i * F::kPitch;
  for (int kb = 0; kb < nkb; ++kb) {
    const bool last = kb + 1 == nkb;
    const uint32_t odd = F::kHalfWord ? (uint32_t(kb) + (odd_rows ? uint32_t(i) : 0u)) & 1u : 0u;
    auto sub = [&](auto sc) __attribute__((always_inline)) {
      constexpr int S = decltype(sc)::value;
      // this step's tokens (at 0 the unit's weights and group sums) have
      // landed; at 3 the next unit's are younger and stay in flight
      if (S == 3 && !last)
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(NW + 2) : "memory");
      else
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if constexpr (S == 0) {
        float ratio[2], mc[2];
        half8 oh[2], ol[2];
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          const uint32_t* row = wrd + 32 * r * F::kPitch;
          const float d = F::dscale(row, odd);
          live[r] = d != 0.f;  // a block of d = 0 has no product terms and keeps the unit
          const float u = live[r] ? d : (unit[r] != 0.f ? unit[r] : 1.f);
          const float inv = __builtin_amdgcn_rcpf(u);
          ratio[r] = unit[r] * inv;
          unit[r] = u;
          oh[r] = F::offsets(row, kg, odd);
          ol[r] = F::offsets(row, kg + 2, odd);
          if constexpr (F::kMin) {
            // the offset products are in units of mscale: into them and back
            const float ms = F::mscale(row);
            mc[r] = ms != 0.f ? ms * inv : 1.f;
            ratio[r] *= __builtin_amdgcn_rcpf(mc[r]);
            if (ms == 0.f) oh[r] = ol[r] = half8{};
          } else if (!live[r]) {
            oh[r] = ol[r] = half8{};
          }
        }
        const uint8_t* sb = sl + i * 64 + kg * 16;
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) {
          const half8 xh = *reinterpret_cast<const half8*>(sb + nb * 2048);
          const half8 xo = *reinterpret_cast<const half8*>(sb + nb * 2048 + 32);
#pragma unroll
          for (int r = 0; r < 2; ++r) {
            acc[r][nb] *= ratio[r];
            acc[r][nb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xo, ol[r], acc[r][nb], 0, 0, 0);
            acc[r][nb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xh, oh[r], acc[r][nb], 0, 0, 0);
            if constexpr (F::kMin) acc[r][nb] *= mc[r];
            __builtin_amdgcn_sched_barrier(0);
          }
        }
#pragma unroll
        for (int r = 0; r < 2; ++r)
          w[r].template load<0>(wrd + 32 * r * F::kPitch, kg, odd, live[r]);
      }
      if constexpr (S == 2) {
#pragma unroll
        for (int r = 0; r < 2; ++r)
          w[r].template load<1>(wrd + 32 * r * F::kPitch, kg, odd, live[r]);
        // the words are in registers: the region is free for the next unit
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      }
      sub128<Q, NMAT, S>(w, xin + (size_t(kb) * 4 + S + 1) * 128, xsrc, xon, S < 3 || !last,
                         xw + ((S & 1) ^ 1) * XBUF, xin + size_t(kb + 1) * 64, ssrc, sw, ws0, ws1,
                         row_bytes, (kb & 1) ? woff0 : woff1, kb + 1, !last, odd_rows, lrow, wl,
                         xl + (S & 1) * XBUF, xoff, acc);
    };
    sub(std::integral_constant<int, 0>{});
    sub(std::integral_constant<int, 1>{});
    sub(std::integral_constant<int, 2>{});
    sub(std::integral_constant<int, 3>{});
  }

  // sum v of lane (i, kg): token 8 (v / 4) + 4 kg + v % 4 of its 32-token
  // block, row i of its 32-row block
  const int ip = (i & ~3) | ((i & 1) << 1) | ((i >> 1) & 1);
#pragma unroll
  for (int nb = 0; nb < 4; ++nb) {
#pragma unroll
    for (int v4 = 0; v4 < 4; ++v4) {
      uint32_t asg[4];
      float wt[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const uint32_t c = min(c0 + uint32_t(32 * nb + 8 * v4 + 4 * kg + v), c1 - 1);
        asg[v] = p.sorted ? p.sorted[c] : c;
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) wt[v] = (NMAT == 2 && p.route_w) ? p.route_w[asg[v]] : 1.0f;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const bool on = c0 + uint32_t(32 * nb + 8 * v4 + 4 * kg + v) < c1;
        if constexpr (NMAT == 2) {
          const float g = acc[0][nb][4 * v4 + v] * unit[0], u = acc[1][nb][4 * v4 + v] * unit[1];
          const _Float16 h = (_Float16)(silu(g) * u * wt[v]);
          uint16_t* row = p.h_out + size_t(asg[v]) * f16_pitch(p.N);
          if (on) row[n0 + ip] = __builtin_bit_cast(uint16_t, h);
          float t = (float)h;  // the sums of the block's two groups of 16 rows
#pragma unroll
          for (int o = 1; o < 16; o <<= 1) t += __shfl_xor(t, o, 16);
          if (on && (i & 15) < 2)
            row[f16_sum_at(p.N, (n0 + i) / 16, i & 1)] = f16_sum_term(t, i & 1);
        } else if (on) {
#pragma unroll
          for (int r = 0; r < 2; ++r)
            p.y_out[size_t(asg[v]) * p.N + n0 + 32 * r + i] = acc[r][nb][4 * v4 + v] * unit[r];
        }
      }
    }
  }
}

}  // namespace grouped
}  // namespace inferno
