// Configuration and launch of the mid-size W4A16 GEMM (kernel: pq_w4a16_mid.h).
#include "pq_w4a16_mid.h"

namespace {

// RB x NT tiles of 16 x 16 per wave, WK waves along K, WN along n; the cost of
// a round of `slots` workgroups (the most the chip holds at once), fitted to
// launches of one full round at K = 4096 (M = 64, 96, 128, 200, 512 at N = 4096:
// 7.7, 9.3, 11.6, 17.7 and 29.5 us, 4.2 us of each fixed).  Small workgroups
// replace each other as they finish, so theirs is paid in part rounds.
struct Cfg {
  int rb, nt, wk, wn, cost, slots;
  bool parts;
};
constexpr Cfg kCfgs[] = {
    {2, 1, 8, 1, 60, 256, false},  {2, 2, 8, 1, 87, 256, false},  {2, 4, 8, 1, 170, 256, false},
    {3, 2, 8, 1, 127, 256, false}, {4, 2, 8, 1, 165, 256, false}, {4, 2, 4, 2, 330, 256, false},
    {4, 2, 2, 4, 660, 256, false}, {2, 2, 4, 1, 260, 768, true},
};

int choose(const pqw16::W16Group& grp, int m) {
  const int nrb = (m + 15) / 16;
  int best = 0;
  double best_cost = 0.0;
  for (int i = 0; i < static_cast<int>(sizeof(kCfgs) / sizeof(kCfgs[0])); ++i) {
    const Cfg& c = kCfgs[i];
    int64_t units = 0;
    for (int q = 0; q < grp.count; ++q) units += (grp.mem[q].n / 16 + c.nt * c.wn - 1) / (c.nt * c.wn);
    const int64_t wgs = units * ((nrb + c.rb - 1) / c.rb);
    const double rounds = c.parts ? static_cast<double>(wgs < c.slots ? c.slots : wgs) / c.slots
                                  : static_cast<double>((wgs + c.slots - 1) / c.slots);
    if (i == 0 || rounds * c.cost < best_cost) {
      best = i;
      best_cost = rounds * c.cost;
    }
  }
  return best;
}

}  // namespace

namespace pqw16 {

// From 17 rows (the decode kernel below streams the weights once) with a group
// of K per wave, while the outputs number at most 2.4 M, or 3.2 M for a group,
// which the prefill tiles run as a launch per member (prefill tiles -> here, us,
// weights from HBM: N = 4096, K = 4096 M = 17 24.8 -> 6.1, 64 25.1 -> 7.7, 200 25.5
// -> 18.4, 512 41.4 -> 29.5; K = 12288 M = 17 68.5 -> 13.7, 200 70.4 -> 44.1; N =
// 12288 M = 128 41.5 -> 28.8, 200 42.7 against 45.0; two of them M = 17 50.7 ->
// 18.1, 128 83 -> 52, 320 113 / 112).  The reads of the larger sizes belong to
// LDS tiles shared by a workgroup.
bool w16_mid_takes(const W16Group& grp, int64_t m, int64_t k) {
  int64_t n = 0;
  for (int i = 0; i < grp.count; ++i) n += grp.mem[i].n;
  return m > 16 && m <= 512 && k >= 1024 && (m + 15) / 16 * 16 * n <= (grp.count > 1 ? 3200000 : 2400000);
}

void launch_w16_mid(const W16Group& grp, int bias_dtype, int y_dtype, int m, int k, hipStream_t stream) {
  switch (choose(grp, m)) {
    case 0: pqmid::launch_w16_mid_t<2, 1, 8, 1>(grp, bias_dtype, y_dtype, m, k, stream); break;
    case 1: pqmid::launch_w16_mid_t<2, 2, 8, 1>(grp, bias_dtype, y_dtype, m, k, stream); break;
    case 2: pqmid::launch_w16_mid_t<2, 4, 8, 1>(grp, bias_dtype, y_dtype, m, k, stream); break;
    case 3: pqmid::launch_w16_mid_t<3, 2, 8, 1>(grp, bias_dtype, y_dtype, m, k, stream); break;
    case 4: pqmid::launch_w16_mid_t<4, 2, 8, 1>(grp, bias_dtype, y_dtype, m, k, stream); break;
    case 5: pqmid::launch_w16_mid_t<4, 2, 4, 2>(grp, bias_dtype, y_dtype, m, k, stream); break;
    case 6: pqmid::launch_w16_mid_t<4, 2, 2, 4>(grp, bias_dtype, y_dtype, m, k, stream); break;
    default: pqmid::launch_w16_mid_t<2, 2, 4, 1>(grp, bias_dtype, y_dtype, m, k, stream); break;
  }
}

}  // namespace pqw16
