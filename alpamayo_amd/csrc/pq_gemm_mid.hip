// Configuration and launch of the mid-size GEMM (kernel: pq_gemm_mid.h).
#include "pq_gemm_mid.h"

namespace {

// A workgroup is 8 waves, one workgroup per CU (its registers): WK waves
// split K, WN sit side by side along n, each on RB x NT tiles of 16 x 16.
struct MidCfg {
  int rb, nt, wk, wn;
};

// The configuration that leaves the busiest CU the least to do.  A wave's
// cost per 128-group, in VALU instructions: 34 to unpack and prepare a 16-column
// tile, 8 to convert and scale a 16 x 16 block; a workgroup's cost is that
// times the groups each wave walks (G / WK, written as 8 / WK since G is
// common to all), and the launch takes ceil(workgroups / 256) of them.  Ties
// go to more columns per workgroup (fewer partial sums through LDS).  One
// column tile per wave where two would leave CUs idle (up to 128 rows).
// Past kMidFixedRows rows WK is gemm_mid_waves(m).
// Measured against the row-major 16-row-block kernel and the LDS-tile kernel,
// weights from HBM (us, before -> after):
//   N = 4096, K = 4096:   M = 32 7.5 -> 5.5, 64 12.5 -> 6.4, 128 18.1 -> 8.1, 200 18.5 -> 11.4, 512 24.6 -> 20.4
//   N = 4096, K = 12288:  M = 32 16.3 -> 11.8, 64 30.1 -> 13.7, 128 47.7 -> 18.9, 200 48.0 -> 27.4, 512 64.9 -> 52.3
//   N = 6144, K = 4096:   M = 32 7.9 -> 7.2, 64 14.9 -> 9.9, 200 24.2 -> 17.1, 320 24.6 -> 22.9
//   N = 24576, K = 4096:  M = 32 19.0 -> 16.7, 64 41.3 -> 22.1, 96 35.3 -> 30.9
MidCfg choose_mid(const pq::GemmGroup& grp, int m) {
  const int nrb = (m + 15) / 16;
  MidCfg best{0, 0, 0, 0};
  int64_t best_cost = 0;
  auto consider = [&](int rb, int nt, int wn) {
    if (m > pq::kMidFixedRows && 8 / wn != pq::gemm_mid_waves(m)) return;
    int64_t units = 0;
    for (int i = 0; i < grp.count; ++i) units += (grp.mem[i].n / 16 + nt * wn - 1) / (nt * wn);
    const int64_t wgs = units * ((nrb + rb - 1) / rb);
    const int64_t cost = (wgs + 255) / 256 * wn * nt * (34 + 8 * rb);
    if (best.rb == 0 || cost < best_cost) {
      best = {rb, nt, 8 / wn, wn};
      best_cost = cost;
    }
  };
  for (int wn = 4; wn >= 1; wn >>= 1) {
    if (m > pq::kMidFixedRows && wn < 4) consider(3, 4, wn);
    for (int rb = 2; rb <= 4; ++rb) consider(rb, 2, wn);
  }
  consider(2, 1, 1);
  return best;
}

template <bool PARTIALS>
void launch_mid(const pq::GemmGroup& grp, int bias_dtype, int y_dtype, int m, int k, hipStream_t s) {
  const MidCfg c = choose_mid(grp, m);
  // weights that one row tile reads once are loaded non-temporally (N = 24576, M = 48: 20.5 -> 19.9 us)
  const bool once = (m + 15) / 16 <= c.rb;
#define PQ_MID(RB_, NT_, WK_, WN_)                                                                             \
  if (c.rb == RB_ && c.nt == NT_ && c.wk == WK_ && c.wn == WN_) {                                              \
    if (!PARTIALS && once)                                                                                     \
      pqmid::launch_mid_t<RB_, NT_, WK_, WN_, !PARTIALS, PARTIALS>(grp, bias_dtype, y_dtype, m, k, s);         \
    else                                                                                                       \
      pqmid::launch_mid_t<RB_, NT_, WK_, WN_, false, PARTIALS>(grp, bias_dtype, y_dtype, m, k, s);             \
    return;                                                                                                    \
  }
  PQ_MID(2, 1, 8, 1)
  PQ_MID(2, 2, 8, 1) PQ_MID(2, 2, 4, 2) PQ_MID(2, 2, 2, 4)
  PQ_MID(3, 2, 8, 1) PQ_MID(3, 2, 4, 2) PQ_MID(3, 2, 2, 4)
  PQ_MID(4, 2, 8, 1) PQ_MID(4, 2, 4, 2) PQ_MID(4, 2, 2, 4)
  PQ_MID(3, 4, 8, 1) PQ_MID(3, 4, 4, 2)
#undef PQ_MID
}

__global__ __launch_bounds__(256) void untile_a_kernel(const int8_t* __restrict__ tiled, int8_t* __restrict__ out,
                                                       int m, int k) {
  const int c16 = k >> 4;
  const int64_t e = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (e >= static_cast<int64_t>(m) * c16) return;
  const int64_t row = e / c16;
  const int kk = static_cast<int>(e - row * c16) * 16;
  *reinterpret_cast<uint4*>(out + row * k + kk) =
      *reinterpret_cast<const uint4*>(tiled + pqd::a_tile_offset(row, kk, m, k >> 7));
}

}  // namespace

namespace pq {

// From 17 rows (below, the decode kernel's one row block streams the weights
// as fast on row-major A) to kMidMaxRows, with at least 8 groups of K, one per
// wave.  Past 2.8 M outputs, 11 K per CU, the LDS tiles of the prefill kernel,
// which share each operand over a workgroup, win where 128 x 256 tiles fill
// half of the CUs, and past 3.2 M outputs its 128 x 128 tiles (N = 24576: M = 96 30.9 against 35.3 us, M = 128 35.2
// against 32.4, M = 200 53 against 42; N = 4096, K = 4096: M = 512 20.4
// against 24.6, M = 800 33 against 31).
MidGemm gemm_mid_choice(const GemmGroup& grp, int64_t m, int64_t k) {
  if (m <= 16 || m > kMidMaxRows || k < 1024) return MidGemm::kNone;
  int64_t n = 0, tiles256 = 0;
  for (int i = 0; i < grp.count; ++i) {
    n += grp.mem[i].n;
    tiles256 += (grp.mem[i].n + 255) / 256;
  }
  const int64_t outputs = (m + 15) / 16 * 16 * n;
  if (gemm_mid_waves(m) == kMidChains && m > kMidFixedRows && outputs > 2800000 &&
      ((m + 127) / 128 * tiles256 >= 128 || outputs > 3200000))
    return MidGemm::kChains;
  return MidGemm::kTiled;
}

void launch_gemm_mid(const GemmGroup& grp, int bias_dtype, int y_dtype, int m, int k, hipStream_t stream) {
  launch_mid<false>(grp, bias_dtype, y_dtype, m, k, stream);
}

void launch_gemm_mid_partials(const GemmGroup& grp, int m, int k, hipStream_t stream) {
  launch_mid<true>(grp, 0, 0, m, k, stream);
}

void launch_untile_a(const int8_t* tiled, int8_t* out, int m, int k, hipStream_t stream) {
  const int64_t chunks = static_cast<int64_t>(m) * (k >> 4);
  untile_a_kernel<<<static_cast<unsigned>((chunks + 255) / 256), 256, 0, stream>>>(tiled, out, m, k);
}

}  // namespace pq
