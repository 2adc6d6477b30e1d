// Host-side check of the addresses of the grouped GEMM's LDS DMA
// (grouped_gemm.hpp): for every format, row width and wavefront, the copies
// of each super-block are replayed from the kernel's own source offsets
// (WSrc) and LDS destinations. Checked: every source piece lies inside the
// expert matrices and is aligned to the piece; lane offsets stay far below
// 2^32; each LDS word of a row is written exactly once and holds the word of
// the row's super-block that W<Q>::load expects there (2 bytes low for a
// half-word super-block of odd index). Prints "OK <n>"; no GPU call.
#include <cstdio>
#include <vector>

#include "grouped_gemm.hpp"

using namespace inferno;
using namespace inferno::grouped;

template <int Q, int RB>
bool check(int N, int nkb) {
  using F = W<Q>;
  constexpr int RPI = WSrc<Q>::RPI, RM = 16 * RB, NI = (RM + RPI - 1) / RPI;
  const int64_t row_bytes = int64_t(nkb) * F::kBytes, total = N * row_bytes;
  const bool odd_rows = F::kHalfWord && (nkb & 1);
  for (int n0 = 0; n0 < N; n0 += RM)
    for (int kb = 0; kb < nkb; ++kb) {
      std::vector<int64_t> lds(size_t(RM) * F::kPitch, -1);
      for (int q = 0; q < NI; ++q)
        for (int lane = 0; lane < 64; ++lane) {
          const int lrow = lane / F::kLanes;
          if (!(lrow < RPI && q * RPI + lrow < RM)) continue;
          const uint32_t o = WSrc<Q>::lane_off(lane, kb & 1, odd_rows, uint32_t(row_bytes));
          const int64_t a = n0 * row_bytes + WSrc<Q>::base(q, kb, odd_rows, row_bytes) + int64_t(o);
          if (o > (1u << 30) || a < 0 || a + F::kChunk > total || a % F::kChunk) {
            std::printf("FAIL: quant %d N %d nkb %d n0 %d kb %d q %d lane %d: source %lld\n", Q, N,
                        nkb, n0, kb, q, lane, (long long)a);
            return false;
          }
          for (int b = 0; b < F::kChunk; b += 4) {
            const size_t w = size_t(q * RPI * F::kPitch) + size_t(lane * F::kChunk + b) / 4;
            if (w >= lds.size() || lds[w] != -1) {
              std::printf("FAIL: quant %d LDS word %zu\n", Q, w);
              return false;
            }
            lds[w] = a + b;
          }
        }
      for (int r = 0; r < RM; ++r) {
        const int odd = F::kHalfWord ? (kb + (odd_rows ? (r & 15) : 0)) & 1 : 0;
        const int64_t block = (n0 + r) * row_bytes + int64_t(kb) * F::kBytes;
        for (int w = 0; w < F::kPitch; ++w)
          if (lds[size_t(r) * F::kPitch + w] != block - 2 * odd + 4 * w) {
            std::printf("FAIL: quant %d nkb %d kb %d row %d word %d\n", Q, nkb, kb, n0 + r, w);
            return false;
          }
        if (4 * F::kPitch < F::kBytes + 2 * odd) return false;
      }
    }
  return true;
}

int main() {
  int n = 0;
  for (int nkb = 1; nkb <= 27; ++nkb)
    for (int N : {128, 256}) {
      if (!check<INFERNO_Q2_K, 2>(N, nkb) || !check<INFERNO_Q2_K, 4>(N, nkb) ||
          !check<INFERNO_Q3_K, 2>(N, nkb) || !check<INFERNO_Q3_K, 4>(N, nkb) ||
          !check<INFERNO_Q4_K, 2>(N, nkb) || !check<INFERNO_Q4_K, 4>(N, nkb) ||
          !check<INFERNO_Q6_K, 2>(N, nkb))
        return 1;
      n += 7;
    }
  std::printf("OK %d\n", n);
  return 0;
}
