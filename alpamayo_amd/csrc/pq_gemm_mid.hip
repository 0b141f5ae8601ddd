// Configuration and launch of the mid-size GEMM (kernel: pq_gemm_mid.h).
#include "pq_gemm_mid.h"

namespace {

// A workgroup is 8 waves, one workgroup per CU (its registers): WK waves
// split K, WN sit side by side along n, each on RB x NT tiles of 16 x 16.
struct MidCfg {
  int rb, nt, wk, wn;
  int64_t cost;   // the busiest CU's, in VALU instructions per wave and 8 groups of K
};

// The configuration that leaves the busiest CU the least to do.  A wave's
// cost per 128-group, in VALU instructions: 34 to unpack and prepare a 16-column
// tile, 8 to convert and scale a 16 x 16 block; a workgroup's cost is that
// times the groups each wave walks (G / WK, written as 8 / WK since G is
// common to all), and the launch takes ceil(workgroups / 256) of them.  Ties
// go to more columns per workgroup (fewer partial sums through LDS).  One
// column tile per wave where two would leave CUs idle (eight waves along K).
// Past kMidFixedRows rows WK is gemm_mid_waves(m, k).
// Measured against the row-major 16-row-block kernel and the LDS-tile kernel,
// weights from HBM (us, before -> after):
//   N = 4096, K = 4096:   M = 32 7.5 -> 5.5, 64 12.5 -> 6.4, 128 18.1 -> 8.1, 200 18.5 -> 11.4
//   N = 4096, K = 12288:  M = 32 16.3 -> 11.8, 64 30.1 -> 13.7, 128 47.7 -> 18.9, 200 48.0 -> 27.4, 512 64.9 -> 52.3
//   N = 6144, K = 4096:   M = 32 7.9 -> 7.2, 64 14.9 -> 9.9, 200 24.2 -> 17.1
//   N = 24576, K = 4096:  M = 32 19.0 -> 16.7, 64 41.3 -> 22.1, 96 35.3 -> 30.9
MidCfg choose_mid(const pq::GemmGroup& grp, int m, int k) {
  const int nrb = (m + 15) / 16;
  MidCfg best{0, 0, 0, 0, 0};
  auto consider = [&](int rb, int nt, int wn) {
    if (m > pq::kMidFixedRows && 8 / wn != pq::gemm_mid_waves(m, k)) return;
    int64_t units = 0;
    for (int i = 0; i < grp.count; ++i) units += (grp.mem[i].n / 16 + nt * wn - 1) / (nt * wn);
    const int64_t wgs = units * ((nrb + rb - 1) / rb);
    const int64_t cost = (wgs + 255) / 256 * wn * nt * (34 + 8 * rb);
    if (best.rb == 0 || cost < best.cost) best = {rb, nt, 8 / wn, wn, cost};
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
  const MidCfg c = choose_mid(grp, m, k);
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

// 17 to 64 rows (else the decode kernel's row blocks on row-major codes): from 16 groups of K on, and past 32 rows
// from 12, or from 8 for up to 16384 columns.  On fewer the final sum over the waves costs more than the order of the
// codes saves (us with the rotation, weights from HBM, decode kernel / here: M = 24, N = 12288 K = 1024 8.8 / 11.3, K =
// 1536 9.9 / 11.8, K = 2048 13.4 / 13.1; M = 64, N = 24576 K = 1024 17.3 / 19.6, K = 2048 25.7 / 23.4).
//
// Past 64 rows whichever of the mid-size GEMM (0.001 us per unit of cost and group of K) and the prefill tiles in its
// order is estimated faster: with few column units the former leaves CUs idle in its last round, with many the
// latter's LDS tiles share each operand over a workgroup (us with the rotation, K = 4096, two members, mid-size / in
// chains / launch_gemm_group's prefill: M = 112 N = 12288 46.8 / 39.1 / 37.2, N = 8192 34.4 / 29.0 / 30.6; M = 144 N =
// 8192 42.0 / 45.7 / 51.5; M = 224 N = 8192 59.0 / 47.4 / 51.7, N = 12288 81.6 / 58.1 / 54.4).
MidGemm gemm_mid_choice(const GemmGroup& grp, int64_t m, int64_t k) {
  if (m <= 16 || k < 1024) return MidGemm::kNone;
  int64_t n = 0;
  for (int i = 0; i < grp.count; ++i) n += grp.mem[i].n;
  if (m <= kMidFixedRows)
    return k >= 2048 || (m > 32 && (k >= 1536 || n <= 16384)) ? MidGemm::kTiled : MidGemm::kNone;
  const int waves = gemm_mid_waves(m, k);
  if (waves != kMidChains) return waves != 0 ? MidGemm::kTiled : MidGemm::kNone;
  const int64_t cost = choose_mid(grp, static_cast<int>(m), static_cast<int>(k)).cost * (k / 128);
  return 0.001 * static_cast<double>(cost) <= gemm_chains_us(grp, m, k) ? MidGemm::kTiled : MidGemm::kChains;
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
