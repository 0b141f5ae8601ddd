// Register-chain rotation from the raw operands (pair indices, angles), for
// many rows: a workgroup owns a 128-channel chunk (one group of 128 or two of
// 64) and a slice of the rows, derives the chunk's chain once and then rotates
// its rows in registers, one cross-lane fetch per layer and row.
//
// The tile form (rotate_kernel in pq_rotate.hip) moves both values of every
// pair through LDS in every layer, 16 bytes per lane at channels that are
// random within the chunk: 2.5 to 3 times the LDS time of a conflict-free
// access, which bounded it, and each workgroup's cos/sin (float64) served 16
// rows only.
//
// The chain: lane l starts with channels l and l + 64 (a matching like any
// layer's) and before every layer keeps one channel and fetches the partner of
// it from the lane that gives it away, so a consistent chain is, for each
// pair of consecutive matchings M, M', a set of kept channels that meets every
// pair of M and of M' once.  M and M' together form even cycles; the two
// orbits of M' M on a cycle are the two alternating halves, and the half with
// the smaller least channel is kept (least channels by pointer doubling).
//
// Bound, forward: the cross-lane fetches (eight per row and chunk, random
// lanes: conflicts in the LDS crossbar) and 65 cycles of VALU a row, 85 cycles
// a row and chunk per CU together; 8192 x 4096 float32 58 us against 102 us on
// the tile form (4.6 TB/s), 2100 x 4096 fp16 in two groups of 64 25.5 -> 18.5 us
// with the operation around it.  Eight waves per workgroup, two workgroups per
// CU: a chain is derived (about 4 us, half of it the float64 sines) once per
// workgroup; four waves and five workgroups took 23.9 us where this takes 21.1.
// Backward: two waves per SIMD (the layers' outputs of four rows are 64
// registers), 8192 x 4096 float32 with both reductions 221 -> 106 us.
//
// Indices that do not pair every channel of a group once (the tile form gives
// them a result too, if an arbitrary one) are detected and take the tile form
// here as well, in the same LDS operations as rotate_kernel.
#pragma once

#include "pq_device.h"
#include "pq_internal.h"

namespace pqchain {

constexpr int kWaves = 8;       // waves per workgroup of the chain kernels
constexpr int kTileWaves = 4;   // and of the tile form of the backward
constexpr int kRows = 4;   // rows per wave and step: a float4 per channel

// One byte per layer of a lane's operands.
template <int KROT>
struct Bytes {
  uint32_t w[(KROT + 3) / 4];
  __device__ __forceinline__ uint32_t get(int r) const { return (w[r >> 2] >> (8 * (r & 3))) & 0xffu; }
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int i = 0; i < (KROT + 3) / 4; ++i) w[i] = 0;
  }
  __device__ __forceinline__ void set(int r, uint32_t v) { w[r >> 2] |= v << (8 * (r & 3)); }
};

template <int KROT, int W = kWaves>
struct Tables {
  static constexpr int kSteps = (KROT + W - 1) / W;   // chain steps per wave (build_tables)
  float2 cs[KROT][64];                         // cos, sin of pair p in layer r
  uint32_t ij[KROT][64];                       // its channels, i | j << 8
  // of each channel: partner | pair << 8 | second of its pair << 14 | whether
  // the partner stays in its lane for the next layer << 15; 0xffff: in no pair
  uint16_t chan[KROT][128];
  uint8_t keep0[128];                          // whether the channel stays in its first lane for layer 0
  union {
    uint16_t scratch[W][kSteps][128];
    uint8_t lane_of[W][KROT][128];
  };
  int bad;
};

template <int KROT>
struct Lane {
  float c[KROT], s[KROT];   // s negated where slot a is the pair's second channel
  Bytes<KROT> src;          // lane to fetch from | 128 when the fetched value goes into slot a
  Bytes<KROT> back;         // lane that fetches from this one
  Bytes<KROT> pr;           // pair index | 128 when slot a is the pair's second channel
  bool swapped;             // slot a starts with channel l + 64
  int fa, fb;               // channels in slots a, b after the last layer
};

// cos, sin and indices of the chunk's 64 pairs per layer: group-local indices
// masked to the group, cos / sin of the stored angle in float64 rounded once
// (as rotate_kernel and the packed operands have them).  A pair past h (the
// empty half of a 64-channel tail) is the identity on two channels of its own.
// All threads; ends with a barrier.  CHAIN: also check them and derive the kept channels.
template <int DT, int KROT, int W, bool CHAIN>
__device__ __forceinline__ void build_tables(Tables<KROT, W>& t, const int16_t* __restrict__ idx,
                                             const void* __restrict__ theta, int h, int G, int chunk) {
  constexpr int NT = W * 64;
  const int half = h >> 1, ch0 = chunk * 128;
  for (int e = threadIdx.x; CHAIN && e < KROT * 128; e += NT) t.chan[e >> 7][e & 127] = 0xffff;
  if (threadIdx.x == 0) t.bad = 0;
  __syncthreads();
  for (int e = threadIdx.x; e < KROT * 64; e += NT) {
    const int r = e >> 6, p = e & 63;
    const int P = chunk * 64 + p;
    float c = 1.0f, sn = 0.0f;
    int i = 2 * p, j = 2 * p + 1;
    if (P < half) {
      const int gi = P / (G / 2);
      const int pp = P % (G / 2);
      const int base = gi * G - ch0;
      const int64_t o = static_cast<int64_t>(r) * h + gi * G + 2 * pp;
      i = base + (idx[o] & (G - 1));
      j = base + (idx[o + 1] & (G - 1));
      const float th = pq_load_as_f32<DT>(theta, static_cast<int64_t>(r) * half + P);
      double sd, cd;
      sincos(static_cast<double>(th), &sd, &cd);
      c = static_cast<float>(cd);
      sn = static_cast<float>(sd);
    }
    t.cs[r][p] = make_float2(c, sn);
    t.ij[r][p] = static_cast<uint32_t>(i) | (static_cast<uint32_t>(j) << 8);
    t.chan[r][i] = static_cast<uint16_t>(j | (p << 8));
    t.chan[r][j] = static_cast<uint16_t>(i | (p << 8) | (1 << 14));
  }
  __syncthreads();
  if constexpr (!CHAIN) return;
  // 64 pairs that reach all 128 channels reach each of them once
  for (int e = threadIdx.x; e < KROT * 128; e += NT)
    if (t.chan[e >> 7][e & 127] == 0xffff) t.bad = 1;
  __syncthreads();
  if (t.bad) return;   // uniform

  // Kept channels of the step into layer r (from layer r - 1, or from the
  // initial pairs x, x ^ 64): least channel of the orbit of
  // x -> M_r(M_{r-1}(x)), at most 64 long, by six doublings.  Wave w takes
  // steps w, w + W, ... side by side (their LDS round trips overlap).
  constexpr int S = Tables<KROT, W>::kSteps;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  uint32_t v[S][2];   // jump target | least channel so far << 8
  int bf[S][2];       // M_{r-1}(x)
#pragma unroll
  for (int q = 0; q < S; ++q) {
    const int r = w + q * W;
    if (r < KROT) {
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int x = lane + 64 * e;
        bf[q][e] = r == 0 ? x ^ 64 : t.chan[r == 0 ? 0 : r - 1][x] & 127;
        v[q][e] = (t.chan[r][bf[q][e]] & 127u) | (static_cast<uint32_t>(x) << 8);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        bf[q][e] = lane;
        v[q][e] = lane;
      }
    }
  }
#pragma unroll
  for (int d = 0; d < 7; ++d) {   // the last exchange leaves the least channels for the comparison below
#pragma unroll
    for (int q = 0; q < S; ++q) {
      t.scratch[w][q][lane] = static_cast<uint16_t>(v[q][0]);
      t.scratch[w][q][lane + 64] = static_cast<uint16_t>(v[q][1]);
    }
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    if (d == 6) break;
#pragma unroll
    for (int q = 0; q < S; ++q)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const uint32_t o = t.scratch[w][q][v[q][e] & 0xff];
        v[q][e] = (o & 0xff) | (min(v[q][e] >> 8, o >> 8) << 8);
      }
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
  }
  // (the other steps read partners and pairs only, which these updates leave as they are)
#pragma unroll
  for (int q = 0; q < S; ++q) {
    const int r = w + q * W;
    if (r < KROT) {
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const uint32_t keep = (v[q][e] >> 8) < (static_cast<uint32_t>(t.scratch[w][q][bf[q][e]]) >> 8) ? 1 : 0;
        if (r == 0) t.keep0[lane + 64 * e] = static_cast<uint8_t>(keep);
        else t.chan[r == 0 ? 0 : r - 1][bf[q][e]] |= static_cast<uint16_t>(keep << 15);
      }
    }
  }
  __syncthreads();
}

// The lane's chain (every wave derives the same one, in its own scratch).
template <int KROT, bool BACK, int W>
__device__ __forceinline__ void build_lane(Tables<KROT, W>& t, Lane<KROT>& p) {
  const int lane = threadIdx.x & 63;
  uint8_t(*lo)[128] = t.lane_of[threadIdx.x >> 6];
  p.src.clear();
  p.back.clear();
  p.pr.clear();
  // the channel given away (slot a) and the one kept (slot b); one lookup per layer on the way
  p.swapped = t.keep0[lane] != 0;
  int a = p.swapped ? lane + 64 : lane, b = a ^ 64;
  uint32_t ent[KROT];
#pragma unroll
  for (int r = 0; r < KROT; ++r) {
    lo[r][a] = static_cast<uint8_t>(lane);
    const uint32_t u = t.chan[r][b];
    ent[r] = u;
    const int partner = u & 127;
    // the fetched channel goes into slot a where it is given away next (anywhere after the last layer)
    const bool into_a = r + 1 < KROT ? (u >> 15) == 0 : true;
    a = into_a ? partner : b;
    b = into_a ? b : partner;
  }
  p.fa = a;
  p.fb = b;
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  uint32_t from[KROT];
#pragma unroll
  for (int r = 0; r < KROT; ++r) from[r] = lo[r][ent[r] & 127];
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  if constexpr (BACK) {
#pragma unroll
    for (int r = 0; r < KROT; ++r) lo[r][from[r]] = static_cast<uint8_t>(lane);   // a lane is fetched from once
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
#pragma unroll
    for (int r = 0; r < KROT; ++r) p.back.set(r, lo[r][lane]);
  }
#pragma unroll
  for (int r = 0; r < KROT; ++r) {
    const uint32_t u = ent[r];
    const bool into_a = r + 1 < KROT ? (u >> 15) == 0 : true;
    // b is the pair's second channel: its partner the first
    const bool b_second = ((u >> 14) & 1) != 0;
    const bool a_second = into_a != b_second;
    const uint32_t pair = (u >> 8) & 63;
    const float2 cs = t.cs[r][pair];
    p.c[r] = cs.x;
    p.s[r] = a_second ? -cs.y : cs.y;
    p.src.set(r, from[r] | (into_a ? 128u : 0u));
    if constexpr (BACK) p.pr.set(r, pair | (a_second ? 128u : 0u));
  }
}

// Layer r of N rows: the update of the float32 sequence that every rotation kernel shares.
template <int KROT, int N>
__device__ __forceinline__ void layer(const Lane<KROT>& p, int r, float (&a)[N], float (&b)[N]) {
  const uint32_t st = p.src.get(r);
  const int addr = static_cast<int>(st & 63u) << 2;
  const bool fl = (st & 128u) != 0;
#pragma unroll
  for (int n = 0; n < N; ++n) {
    const float recv = __int_as_float(__builtin_amdgcn_ds_bpermute(addr, __float_as_int(a[n])));
    const float keep = b[n];
    const float u = fl ? recv : keep, v = fl ? keep : recv;
    pqd::givens(u, v, p.c[r], p.s[r], a[n], b[n]);
  }
}

// Layer r in the tile form: pair `lane` of four rows through LDS.
template <int KROT, int W>
__device__ __forceinline__ void tile_layer(const Tables<KROT, W>& t, int r, int lane, float4* wt, float4& na, float4& nb) {
  const float2 cs = t.cs[r][lane];
  const uint32_t ij = t.ij[r][lane];
  const int i = static_cast<int>(ij & 0xffu), j = static_cast<int>(ij >> 8);
  const float4 a = wt[i], b = wt[j];
  pqd::givens(a.x, b.x, cs.x, cs.y, na.x, nb.x);
  pqd::givens(a.y, b.y, cs.x, cs.y, na.y, nb.y);
  pqd::givens(a.z, b.z, cs.x, cs.y, na.z, nb.z);
  pqd::givens(a.w, b.w, cs.x, cs.y, na.w, nb.w);
  wt[i] = na;
  wt[j] = nb;
  // the tile is the wave's alone and its LDS operations complete in order;
  // the fence keeps the compiler from moving them
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// Raw values of channels lane and lane + 64 of the chunk in kRows rows from
// `row` (clamped to the last row; channels past h read channel 0 of the chunk).
template <int DT>
__device__ __forceinline__ void load_rows(const void* __restrict__ x, int64_t row, int64_t rows, int h, int ch0, int lane,
                                          uint32_t (&lo)[kRows], uint32_t (&hi)[kRows]) {
  constexpr int kSz = DT == PQ_F32 ? 4 : 2;
  const int c1 = ch0 + 64 < h ? 64 : 0;
#pragma unroll
  for (int q = 0; q < kRows; ++q) {
    const int64_t o = (row + q < rows ? row + q : rows - 1) * h + ch0;   // uniform over the wave
    const char* base = static_cast<const char*>(x) + o * kSz;
    lo[q] = pq_load_raw<DT>(base, lane);
    hi[q] = pq_load_raw<DT>(base, lane + c1);
  }
}

// grid (row slices, chunks).  MX: OCP MXFP4 codes to y and E8M0 scales to sc
// instead of the rotated rows, as rotate_kernel.
template <int DT, int KROT, bool MX>
__global__ __launch_bounds__(kWaves * 64) void rotate_chain(const void* __restrict__ x, void* __restrict__ y,
                                                            uint8_t* __restrict__ sc, const int16_t* __restrict__ idx,
                                                            const void* __restrict__ theta,
                                                            const void* __restrict__ scales, int64_t rows, int h,
                                                            int G, int64_t slice) {
  __shared__ Tables<KROT> t;
  __shared__ float4 tile[kWaves][128];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // wave-uniform rows: scalar addresses
  const int ch0 = blockIdx.y * 128;
  const bool ok1 = ch0 + 64 < h;   // whether the chunk has its second 64 channels
  const int64_t row_end = min(rows, (static_cast<int64_t>(blockIdx.x) + 1) * slice);
  int64_t row = static_cast<int64_t>(blockIdx.x) * slice + w * kRows;
  uint32_t lo[kRows], hi[kRows];
  load_rows<DT>(x, row, rows, h, ch0, lane, lo, hi);
  float s0 = 1.0f, s1 = 1.0f;
  if (scales != nullptr) {
    s0 = pq_load_as_f32<DT>(scales, ch0 + lane);
    s1 = pq_load_as_f32<DT>(scales, ch0 + (ok1 ? 64 : 0) + lane);
  }
  build_tables<DT, KROT, kWaves, true>(t, idx, theta, h, G, blockIdx.y);
  const bool chain = t.bad == 0;
  Lane<KROT> p;
  if (chain) build_lane<KROT, false>(t, p);
  float4* wt = tile[w];
  for (; row < row_end; row += kWaves * kRows) {
    float a[kRows], b[kRows];
#pragma unroll
    for (int q = 0; q < kRows; ++q) {
      a[q] = pq_raw_to_f32<DT>(lo[q]);
      b[q] = ok1 ? pq_raw_to_f32<DT>(hi[q]) : 0.0f;
      if (scales != nullptr) {
        a[q] = a[q] * s0;
        b[q] = b[q] * s1;
      }
    }
    load_rows<DT>(x, row + kWaves * kRows, rows, h, ch0, lane, lo, hi);
    if (chain) {
      float u[kRows], v[kRows];
#pragma unroll
      for (int q = 0; q < kRows; ++q) {
        u[q] = p.swapped ? b[q] : a[q];
        v[q] = p.swapped ? a[q] : b[q];
      }
#pragma unroll
      for (int r = 0; r < KROT; ++r) layer<KROT, kRows>(p, r, u, v);
      wt[p.fa] = make_float4(u[0], u[1], u[2], u[3]);
      wt[p.fb] = make_float4(v[0], v[1], v[2], v[3]);
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
    } else {
      wt[lane] = make_float4(a[0], a[1], a[2], a[3]);
      wt[lane + 64] = make_float4(b[0], b[1], b[2], b[3]);
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      float4 na, nb;
      for (int r = 0; r < KROT; ++r) tile_layer<KROT>(t, r, lane, wt, na, nb);
    }
    const float4 fa = wt[2 * lane], fb = wt[2 * lane + 1];
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    float va[kRows] = {fa.x, fa.y, fa.z, fa.w};
    float vb[kRows] = {fb.x, fb.y, fb.z, fb.w};
    if constexpr (MX) {
      // a 32-channel block = 16 lanes.  The blocks' maxima of all rows by
      // DPP; the magnitudes order like unsigned integers, NaN above
      // infinity, so a NaN shows in the maximum and only then the blocks'
      // flags and NaN-free maxima are formed.
      uint32_t mx[kRows];
#pragma unroll
      for (int q = 0; q < kRows; ++q)
        mx[q] = max(__float_as_uint(va[q]) & 0x7fffffffu, __float_as_uint(vb[q]) & 0x7fffffffu);
      auto block_max = [&](uint32_t (&u)[kRows]) {
#pragma unroll
        for (int q = 0; q < kRows; ++q) u[q] = pq_dpp_umax<0xb1, 0xf>(u[q]);
#pragma unroll
        for (int q = 0; q < kRows; ++q) u[q] = pq_dpp_umax<0x4e, 0xf>(u[q]);
#pragma unroll
        for (int q = 0; q < kRows; ++q) u[q] = pq_dpp_umax<0x141, 0xf>(u[q]);
#pragma unroll
        for (int q = 0; q < kRows; ++q) u[q] = pq_dpp_umax<0x140, 0xf>(u[q]);
      };
      block_max(mx);
      bool nan[kRows];
      bool any = false;
#pragma unroll
      for (int q = 0; q < kRows; ++q) {
        nan[q] = mx[q] > 0x7f800000u;
        any = any || nan[q];
      }
      if (__ballot(any) != 0) {
#pragma unroll
        for (int q = 0; q < kRows; ++q) {
          // a NaN element counts as zero (its block's scale says NaN)
          va[q] = va[q] == va[q] ? va[q] : 0.0f;
          vb[q] = vb[q] == vb[q] ? vb[q] : 0.0f;
          mx[q] = max(__float_as_uint(va[q]) & 0x7fffffffu, __float_as_uint(vb[q]) & 0x7fffffffu);
        }
        block_max(mx);
      }
#pragma unroll
      for (int q = 0; q < kRows; ++q) {
        const int ex = pqd::mx_shared_exp(__uint_as_float(mx[q]));
        const float inv = pqd::mx_inv_scale(ex);
        // both codes, rounded to nearest even and saturated, in the low byte
        const uint32_t code = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(0u, va[q] * inv, vb[q] * inv, 1.0f, 0);
        if (row + q < row_end && 2 * lane < h - ch0) {
          (static_cast<uint8_t*>(y) + (row + q) * (h >> 1) + (ch0 >> 1))[lane] = static_cast<uint8_t>(code);
          if ((lane & 15) == 0)
            (sc + (row + q) * (h >> 5) + (ch0 >> 5))[lane >> 4] = nan[q] ? 0xFFu : static_cast<uint8_t>(ex + 127);
        }
      }
    } else {
#pragma unroll
      for (int q = 0; q < kRows; ++q) {
        if (row + q < row_end) {
          const int64_t o = (row + q) * h + ch0;
          if (2 * lane < h - ch0) {
            if constexpr (DT == PQ_F32) {
              float* d = static_cast<float*>(y) + o;
              d[2 * lane] = va[q];
              d[2 * lane + 1] = vb[q];
            } else {
              uint16_t* d = static_cast<uint16_t*>(y) + o;
              d[2 * lane] = DT == PQ_F16 ? pq_f32_to_f16(va[q]) : pq_f32_to_bf16(va[q]);
              d[2 * lane + 1] = DT == PQ_F16 ? pq_f32_to_f16(vb[q]) : pq_f32_to_bf16(vb[q]);
            }
          }
        }
      }
    }
  }
}

// Gradients (the formulas: pq_rotate_bwd.hip).  Per step of four rows a wave
// re-runs the layers on t = s * x, keeping every layer's outputs (a', b'),
// then walks back on grad_y: with (g_a, g_b) at a layer's outputs the angle
// gradient is g_a b' - g_b a' (negated where slot a is the pair's second
// channel: the lane turns by -theta), the gradient at its inputs the
// transposed turn, and the fetched channel's goes back to the lane it came
// from.  Sums over the rows stay in registers; part_th [nb][KROT][h/2] and
// part_s [nb][h] take one partial per workgroup row.
// grid (nb, chunks); workgroup row b takes the 4 W-row tiles b, b + nb, ...
// CHAIN = false runs the tile form alone (few rows per workgroup).
template <int DT, int KROT, int W, bool CHAIN>
__global__ __launch_bounds__(W * 64) void rotate_chain_bwd(
    const void* __restrict__ x, const void* __restrict__ gy, void* __restrict__ gx, const int16_t* __restrict__ idx,
    const void* __restrict__ theta, const void* __restrict__ scales, float* __restrict__ part_th,
    float* __restrict__ part_s, int64_t rows, int h, int G, int krot) {   // krot = KROT (see the tile form)
  __shared__ Tables<KROT, W> t;
  __shared__ float4 tile[W][128];
  __shared__ float red[W][KROT][64];
  __shared__ float red_s[W][128];
  constexpr int kTile = W * kRows;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // wave-uniform rows: scalar addresses
  const int ch0 = blockIdx.y * 128;
  const bool ok1 = ch0 + 64 < h;
  float s0 = 1.0f, s1 = 1.0f;
  if (scales != nullptr) {
    s0 = pq_load_as_f32<DT>(scales, ch0 + lane);
    s1 = pq_load_as_f32<DT>(scales, ch0 + (ok1 ? 64 : 0) + lane);
  }
  build_tables<DT, KROT, W, CHAIN>(t, idx, theta, h, G, blockIdx.y);
  const bool chain = CHAIN && t.bad == 0;
  Lane<KROT> p;
  if (chain) build_lane<KROT, true>(t, p);
  float4* wt = tile[w];
  // sums of up to eight steps, and of those sums (short chains keep the rounding of thousands of rows small)
  float acc_th[KROT], all_th[KROT];
#pragma unroll
  for (int r = 0; r < KROT; ++r) acc_th[r] = all_th[r] = 0.0f;
  float acc_s0 = 0.0f, acc_s1 = 0.0f, all_s0 = 0.0f, all_s1 = 0.0f;
  int since = 0;
  auto flush = [&]() {
#pragma unroll
    for (int r = 0; r < KROT; ++r) {
      all_th[r] += acc_th[r];
      acc_th[r] = 0.0f;
    }
    all_s0 += acc_s0;
    all_s1 += acc_s1;
    acc_s0 = acc_s1 = 0.0f;
    since = 0;
  };
  const int64_t step = static_cast<int64_t>(gridDim.x) * kTile;
  for (int64_t row = static_cast<int64_t>(blockIdx.x) * kTile + w * kRows; row < rows; row += step) {
    uint32_t lo[kRows], hi[kRows], glo[kRows], ghi[kRows];
    load_rows<DT>(x, row, rows, h, ch0, lane, lo, hi);
    load_rows<DT>(gy, row, rows, h, ch0, lane, glo, ghi);
    float xa[kRows], xb[kRows], ga[kRows], gb[kRows];
#pragma unroll
    for (int q = 0; q < kRows; ++q) {
      const bool live = row + q < rows;   // rows past the end add nothing to the sums
      xa[q] = live ? pq_raw_to_f32<DT>(lo[q]) : 0.0f;
      xb[q] = live && ok1 ? pq_raw_to_f32<DT>(hi[q]) : 0.0f;
      ga[q] = live ? pq_raw_to_f32<DT>(glo[q]) : 0.0f;
      gb[q] = live && ok1 ? pq_raw_to_f32<DT>(ghi[q]) : 0.0f;
    }
    float a[kRows], b[kRows];
#pragma unroll
    for (int q = 0; q < kRows; ++q) {
      a[q] = scales != nullptr ? xa[q] * s0 : xa[q];
      b[q] = scales != nullptr ? xb[q] * s1 : xb[q];
    }
    float ta[kRows], tb[kRows];   // the gradient at t, channels lane and lane + 64
    if (chain) {
      float oa[KROT][kRows], ob[KROT][kRows];
      float u[kRows], v[kRows];
#pragma unroll
      for (int q = 0; q < kRows; ++q) {
        u[q] = p.swapped ? b[q] : a[q];
        v[q] = p.swapped ? a[q] : b[q];
      }
#pragma unroll
      for (int r = 0; r < KROT; ++r) {
        layer<KROT, kRows>(p, r, u, v);
#pragma unroll
        for (int q = 0; q < kRows; ++q) {
          oa[r][q] = u[q];
          ob[r][q] = v[q];
        }
      }
      // grad_y from channel order to the slots of the last layer
      wt[lane] = make_float4(ga[0], ga[1], ga[2], ga[3]);
      wt[lane + 64] = make_float4(gb[0], gb[1], gb[2], gb[3]);
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      const float4 g0 = wt[p.fa], g1 = wt[p.fb];
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      u[0] = g0.x; u[1] = g0.y; u[2] = g0.z; u[3] = g0.w;
      v[0] = g1.x; v[1] = g1.y; v[2] = g1.z; v[3] = g1.w;
#pragma unroll
      for (int r = KROT - 1; r >= 0; --r) {
        const float c = p.c[r], s = p.s[r];
        const bool fl = (p.src.get(r) & 128u) != 0;
        const int addr = static_cast<int>(p.back.get(r)) << 2;
        float d = 0.0f;
#pragma unroll
        for (int q = 0; q < kRows; ++q) {
          const float e = fmaf(u[q], ob[r][q], -(v[q] * oa[r][q]));
          d = q == 0 ? e : d + e;
        }
        acc_th[r] += d;
#pragma unroll
        for (int q = 0; q < kRows; ++q) {
          const float pa = fmaf(u[q], c, -(v[q] * s));
          const float pb = fmaf(v[q], c, u[q] * s);
          // the fetched channel's gradient goes back, the kept one's into slot b
          u[q] = __int_as_float(__builtin_amdgcn_ds_bpermute(addr, __float_as_int(fl ? pa : pb)));
          v[q] = fl ? pb : pa;
        }
      }
#pragma unroll
      for (int q = 0; q < kRows; ++q) {
        ta[q] = p.swapped ? v[q] : u[q];
        tb[q] = p.swapped ? u[q] : v[q];
      }
    } else {
      wt[lane] = make_float4(a[0], a[1], a[2], a[3]);
      wt[lane + 64] = make_float4(b[0], b[1], b[2], b[3]);
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      // alone, with a branch per layer on the run-time count: without it the operands of
      // all layers are read ahead and kept over the row loop, five registers
      // a layer
      float4 oa[KROT], ob[KROT];
#pragma unroll
      for (int r = 0; r < KROT; ++r)
        if (CHAIN || r < krot) tile_layer<KROT>(t, r, lane, wt, oa[r], ob[r]);
      wt[lane] = make_float4(ga[0], ga[1], ga[2], ga[3]);
      wt[lane + 64] = make_float4(gb[0], gb[1], gb[2], gb[3]);
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
#pragma unroll
      for (int r = KROT - 1; r >= 0; --r) {
        if (!CHAIN && r >= krot) continue;
        const float2 cs = t.cs[r][lane];
        const uint32_t ij = t.ij[r][lane];
        const int i = static_cast<int>(ij & 0xffu), j = static_cast<int>(ij >> 8);
        const float4 g0 = wt[i], g1 = wt[j];
        float d = fmaf(g0.x, ob[r].x, -(g1.x * oa[r].x));
        d += fmaf(g0.y, ob[r].y, -(g1.y * oa[r].y));
        d += fmaf(g0.z, ob[r].z, -(g1.z * oa[r].z));
        d += fmaf(g0.w, ob[r].w, -(g1.w * oa[r].w));
        acc_th[r] += d;
        wt[i] = make_float4(fmaf(g0.x, cs.x, -(g1.x * cs.y)), fmaf(g0.y, cs.x, -(g1.y * cs.y)),
                            fmaf(g0.z, cs.x, -(g1.z * cs.y)), fmaf(g0.w, cs.x, -(g1.w * cs.y)));
        wt[j] = make_float4(fmaf(g1.x, cs.x, g0.x * cs.y), fmaf(g1.y, cs.x, g0.y * cs.y),
                            fmaf(g1.z, cs.x, g0.z * cs.y), fmaf(g1.w, cs.x, g0.w * cs.y));
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
      }
      const float4 f0 = wt[lane], f1 = wt[lane + 64];
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      ta[0] = f0.x; ta[1] = f0.y; ta[2] = f0.z; ta[3] = f0.w;
      tb[0] = f1.x; tb[1] = f1.y; tb[2] = f1.z; tb[3] = f1.w;
    }
#pragma unroll
    for (int q = 0; q < kRows; ++q) {
      if (row + q < rows) {
        char* d = static_cast<char*>(gx) + ((row + q) * h + ch0) * (DT == PQ_F32 ? 4 : 2);
        pq_store_from_f32<DT>(d, lane, scales != nullptr ? ta[q] * s0 : ta[q]);
        if (ok1) pq_store_from_f32<DT>(d, lane + 64, scales != nullptr ? tb[q] * s1 : tb[q]);
      }
      if (scales != nullptr) {
        acc_s0 = fmaf(xa[q], ta[q], acc_s0);
        acc_s1 = fmaf(xb[q], tb[q], acc_s1);
      }
    }
    if (++since == 8) flush();
  }
  flush();

  // Sum the waves (fixed order) and write this workgroup's partials.
#pragma unroll
  for (int r = 0; r < KROT; ++r) {
    const uint32_t pr = chain ? p.pr.get(r) : static_cast<uint32_t>(lane);
    red[w][r][pr & 63u] = (pr & 128u) != 0 ? -all_th[r] : all_th[r];
  }
  red_s[w][lane] = all_s0;
  red_s[w][lane + 64] = all_s1;
  __syncthreads();
  const int half = h >> 1;
  for (int e = threadIdx.x; e < KROT * 64; e += W * 64) {
    const int r = e >> 6, P = blockIdx.y * 64 + (e & 63);
    float v = red[0][r][e & 63];
#pragma unroll
    for (int k = 1; k < W; ++k) v += red[k][r][e & 63];
    if (P < half) part_th[(static_cast<int64_t>(blockIdx.x) * KROT + r) * half + P] = v;
  }
  if (scales != nullptr && threadIdx.x < 128 && ch0 + static_cast<int>(threadIdx.x) < h) {
    const int e = threadIdx.x;
    float v = red_s[0][e];
#pragma unroll
    for (int k = 1; k < W; ++k) v += red_s[k][e];
    part_s[static_cast<int64_t>(blockIdx.x) * h + ch0 + e] = v;
  }
}

}  // namespace pqchain
