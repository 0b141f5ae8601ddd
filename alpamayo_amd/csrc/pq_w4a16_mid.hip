// Configuration and launch of the mid-size W4A16 GEMM (kernel: pq_w4a16_mid.h).
#include <algorithm>

#include "pq_w4a16_mid.h"

namespace {

// RB x NT tiles of 16 x 16 per wave, WK waves along K, WN along n; the cost of
// a round of `slots` workgroups (the most the chip holds at once), fitted to
// launches of one full round at K = 4096 (M = 64, 96, 128, 200, 512 at N = 4096:
// 7.7, 9.3, 11.6, 17.7 and 29.5 us, 4.2 us of each fixed).  Small workgroups
// replace each other as they finish, so theirs is paid in part rounds (a fifth
// at least: N = 2 x 6912, K = 4096, M = 33 26.5 us, 22.6 on 3 x 2 blocks), and
// while the fp16 rows fit an XCD's L2 (4 MB: 2 M values) it is 0.83 of what it
// is past that (with the rotation, N = 4096: M = 320, K = 4096 35.2 us against
// 38.6 on eight waves of 2 x 2 blocks; M = 400, K = 12288 108 against 102 on
// the 4 x 2 blocks in two columns).
struct Cfg {
  int rb, nt, wk, wn, cost, slots;
  bool parts;
};
constexpr Cfg kCfgs[] = {
    {2, 1, 8, 1, 60, 256, false},  {2, 2, 8, 1, 87, 256, false},  {2, 4, 8, 1, 170, 256, false},
    {3, 2, 8, 1, 127, 256, false}, {4, 2, 8, 1, 165, 256, false}, {4, 2, 4, 2, 330, 256, false},
    {2, 2, 4, 1, 215, 768, true},
};

struct Choice {
  int cfg;
  double cost;
};

// The cheapest configuration for `count` linears of n[i] columns.
Choice choose(const int* n, int count, int m, int k) {
  const int nrb = (m + 15) / 16;
  Choice best{0, 0.0};
  for (int i = 0; i < static_cast<int>(sizeof(kCfgs) / sizeof(kCfgs[0])); ++i) {
    const Cfg& c = kCfgs[i];
    int64_t units = 0;
    for (int q = 0; q < count; ++q) units += (n[q] / 16 + c.nt * c.wn - 1) / (c.nt * c.wn);
    const int64_t wgs = units * ((nrb + c.rb - 1) / c.rb);
    double rounds = static_cast<double>((wgs + c.slots - 1) / c.slots);
    if (c.parts && wgs > c.slots && wgs % c.slots != 0)
      rounds = static_cast<double>(wgs / c.slots) + std::max(static_cast<double>(wgs % c.slots) / c.slots, 0.2);
    double cost = c.cost * rounds;
    if (c.parts && static_cast<int64_t>(m) * k > 2 << 20) cost *= 1.2;
    if (i == 0 || cost < best.cost) best = {i, cost};
  }
  return best;
}

}  // namespace

namespace pqw16 {

// From 17 rows (the decode kernel below streams the weights once) with a group of K per part, where the linear alone
// is estimated faster here, or two of it in one launch clearly (0.8) faster than in two of the prefill tiles and the
// linear alone not much slower: a group runs what its members run alone (the two GEMMs' MFMAs add in other orders),
// so the choice must not look at the others.  Estimates in us, less the fixed part of a launch here (4.2), fitted to
// launches of 17 to 512 rows at K = 1024 to 12288 with the weights in the caches and from HBM (prefill tiles -> here, us
// with the rotation, weights from HBM: K = 4096, N = 4096 M = 64 35.6 -> 17.8; two of N = 12288 M = 96 105 -> 70).
bool w16_mid_takes(int64_t m, int64_t n, int64_t k) {
  if (m <= 16 || m > 512 || k < 1024) return false;
  const int two[2] = {static_cast<int>(n), static_cast<int>(n)};
  const double per_cost = (k < 2048 ? 0.8 : 1.0) * (0.00118 * static_cast<double>(k / 128) + 0.021);   // FEW below 2048
  const double here = choose(two, 1, static_cast<int>(m), static_cast<int>(k)).cost * per_cost;
  const double here2 = choose(two, 2, static_cast<int>(m), static_cast<int>(k)).cost * per_cost;
  const double there = w16_prefill_us(m, n, k);
  return here < there || (here2 < 0.8 * (2.0 * there + 4.5) && here < 1.2 * there);
}

void launch_w16_mid(const W16Group& grp, int bias_dtype, int y_dtype, int m, int k, hipStream_t stream) {
  int n[pq::kMaxGroup];
  for (int i = 0; i < grp.count; ++i) n[i] = grp.mem[i].n;
  switch (choose(n, grp.count, m, k).cfg) {
    case 0: pqmid::launch_w16_mid_t<2, 1, 8, 1>(grp, bias_dtype, y_dtype, m, k, stream); break;
    case 1: pqmid::launch_w16_mid_t<2, 2, 8, 1>(grp, bias_dtype, y_dtype, m, k, stream); break;
    case 2: pqmid::launch_w16_mid_t<2, 4, 8, 1>(grp, bias_dtype, y_dtype, m, k, stream); break;
    case 3: pqmid::launch_w16_mid_t<3, 2, 8, 1>(grp, bias_dtype, y_dtype, m, k, stream); break;
    case 4: pqmid::launch_w16_mid_t<4, 2, 8, 1>(grp, bias_dtype, y_dtype, m, k, stream); break;
    case 5: pqmid::launch_w16_mid_t<4, 2, 4, 2>(grp, bias_dtype, y_dtype, m, k, stream); break;
    default: pqmid::launch_w16_mid_t<2, 2, 4, 1>(grp, bias_dtype, y_dtype, m, k, stream); break;
  }
}

}  // namespace pqw16
