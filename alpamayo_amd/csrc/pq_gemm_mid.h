// int4-weight x int8-activation GEMM for 17 to a few hundred rows, on tiled A.
//
// Between the decode sizes (every wave streams its weights once, A is tiny)
// and the prefill sizes (big LDS tiles shared by a workgroup) a launch has
// too few big tiles to fill the chip and too many rows for one row block.
// Here a wave owns RB x NT blocks of 16 x 16 outputs and walks one of
// WK parts of K on its own: operands go from memory straight into
// registers, two groups ahead, and no wave waits for another until the WK
// partial sums of a workgroup meet in LDS at the end (added in a fixed
// order).  No barrier in the K loop, so the waves of a SIMD drift apart and
// one's unpacking and scaling (VALU) run under the other's MFMAs.
//
// A comes tiled (pqd::a_tile_offset): the 16 rows x 128 codes of a block are
// stored in the order the MFMA lanes take them, so a fragment is one
// contiguous 1 KB load.  From row-major codes each lane reads 16 bytes of a
// different row, which the L1 serves one lane per cycle.
#pragma once

#include <type_traits>

#include "pq_device.h"
#include "pq_internal.h"

namespace pqmid {

using namespace pqd;

template <int RB, int NT>
struct Stage {
  v4i a[RB][2];
  v4i w[NT];
  uint32_t meta[NT];
};

// A wave-uniform address kept in scalar registers: the lane's part of the
// load address then is one 32-bit offset, where the compiler otherwise walks
// a 64-bit address per lane and operand through the loop (2 (2 RB + 2 NT)
// VGPRs, which spilled the 4 x 4 instance).
template <bool ON, typename T>
__device__ __forceinline__ const uint8_t* scalar_base(const T* p) {
  uint64_t u = reinterpret_cast<uint64_t>(p);
  if constexpr (ON) asm("" : "+s"(u));
  return reinterpret_cast<const uint8_t*>(u);
}

// The member of a group that owns column unit `unit` (wave-uniform).
__device__ __forceinline__ int member_of(const pq::GemmGroup& grp, int unit) {
  int mi = 0;
#pragma unroll
  for (int i = 1; i < pq::kMaxGroup; ++i)
    if (i < grp.count && unit >= grp.first[i]) mi = i;
  return mi;
}

// Partial sums kept in LDS: all of them up to four per column, else half
// (the upper half of the waves hands its sums to the lower half first).
constexpr int kept(int wk) { return wk >= 8 ? wk / 2 : wk; }

template <int RB, int NT, int WK, int WN>
constexpr size_t lds_bytes() { return static_cast<size_t>(kept(WK)) * WN * RB * NT * 4 * 64 * sizeof(float); }

// grid: row tiles x column units (units of NT * WN 16-column tiles; members
// start on a unit).  NTW: the weights are read by one row tile only, so they
// are loaded non-temporally.
template <int RB, int NT, int WK, int WN, bool NTW, bool PARTIALS>
__global__ __launch_bounds__(WK * WN * 64) void gemm_mid(const pq::GemmGroup grp, int bias_dtype, int y_dtype, int M,
                                                         int K) {
  extern __shared__ __attribute__((aligned(16))) float red[];
  const int G = K >> 7;
  const int nrb = (M + 15) >> 4;
  const int nrt = (nrb + RB - 1) / RB;
  // Workgroup b runs on XCD b % 8: each XCD takes a contiguous run of
  // (column unit, row tile) pairs, row tiles innermost, so the row tiles that
  // read the same weights share an L2.
  const int q8 = gridDim.x >> 3, r8 = gridDim.x & 7, xcd = blockIdx.x & 7;
  const int t = xcd * q8 + min(xcd, r8) + (blockIdx.x >> 3);
  const int unit = t / nrt, rt = t - unit * nrt;
  const int mi = member_of(grp, unit);
  const pq::GemmMember& mb = grp.mem[mi];
  const int N = mb.n;
  const int ntiles = N >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wk = wave / WN, wn = wave % WN;
  const int lane = threadIdx.x & 63;
  const int c = lane & 15, j = lane >> 4;
  const int tile0 = (unit - grp.first[mi]) * (NT * WN);   // the workgroup's first 16-column tile

  // Tiles past N and row blocks past M are clamped; their results are not stored.
  const uint8_t* wp[NT];
  const uint32_t* mp[NT];
  const int8_t* ap[RB];
  uint32_t ar[RB], al[RB];   // the block's rows; the lane's part of its fragments
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int64_t o = static_cast<int64_t>(min(tile0 + wn * NT + nt, ntiles - 1)) * G;
    wp[nt] = mb.wpack + o * 1024;
    mp[nt] = mb.wmeta + o * 16;
  }
#pragma unroll
  for (int b = 0; b < RB; ++b) {
    const int rb = min(rt * RB + b, nrb - 1);
    ap[b] = mb.xq + static_cast<int64_t>(rb) * G * 2048;
    ar[b] = min(M - rb * 16, 16);
    al[b] = (j * ar[b] + min(static_cast<uint32_t>(c), ar[b] - 1)) * 16;   // rows past M repeat the last
  }

  const uint32_t l16 = lane * 16, c4 = c * 4;
  auto load = [&](Stage<RB, NT>& s, int g) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const v4i* w = reinterpret_cast<const v4i*>(scalar_base<!PARTIALS>(wp[nt] + g * 1024) + l16);
      const uint32_t* m = reinterpret_cast<const uint32_t*>(scalar_base<!PARTIALS>(mp[nt] + g * 16) + c4);
      s.w[nt] = NTW ? __builtin_nontemporal_load(w) : *w;
      s.meta[nt] = NTW ? __builtin_nontemporal_load(m) : *m;
    }
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      s.a[b][0] = *reinterpret_cast<const v4i*>(scalar_base<!PARTIALS>(ap[b] + 2 * g * 64 * ar[b]) + al[b]);
      s.a[b][1] = *reinterpret_cast<const v4i*>(scalar_base<!PARTIALS>(ap[b] + (2 * g + 1) * 64 * ar[b]) + al[b]);
    }
  };

  float acc[RB][NT][4];
#pragma unroll
  for (int b = 0; b < RB; ++b)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[b][nt][v] = 0.0f;

  auto compute = [&](const Stage<RB, NT>& s, int g) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const uint32_t meta = s.meta[nt];
      const uint32_t zb = meta_zero_bias(meta);
      const v4i w = s.w[nt];
      const v4i b0 = unpack16(static_cast<uint32_t>(w.x), static_cast<uint32_t>(w.y), zb);
      const v4i b1 = unpack16(static_cast<uint32_t>(w.z), static_cast<uint32_t>(w.w), zb);
      const float sc = meta_scale(meta);
      v4i p[RB];
#pragma unroll
      for (int b = 0; b < RB; ++b) p[b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(s.a[b][0], b0, v4i{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
      for (int b = 0; b < RB; ++b) p[b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(s.a[b][1], b1, p[b], 0, 0, 0);
#pragma unroll
      for (int b = 0; b < RB; ++b)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          if constexpr (PARTIALS) {
            const int m = (rt * RB + b) * 16 + 4 * j + v;
            const int tile = tile0 + wn * NT + nt;
            if (m < M && tile < ntiles)
              mb.partials[(static_cast<int64_t>(m) * G + g) * N + tile * 16 + c] = p[b][v];
          } else {
            acc[b][nt][v] = fmaf(static_cast<float>(p[b][v]), sc, acc[b][nt][v]);
          }
        }
    }
  };

  // Wave wk walks the n groups of its part of K (the host keeps WK <= G).
  // Two register stages; the tail is peeled so that no load sits behind a
  // branch (the compiler would wait for every load at the join).
  const int gb = wk * G / WK, n = (wk + 1) * G / WK - gb;
  auto grp_of = [&](int i) { return gb + i; };
  Stage<RB, NT> s0, s1;
  load(s0, grp_of(0));
  load(s1, grp_of(min(1, n - 1)));
  int i = 0;
  for (; i + 3 < n; i += 2) {
    compute(s0, grp_of(i));
    load(s0, grp_of(i + 2));
    compute(s1, grp_of(i + 1));
    load(s1, grp_of(i + 3));
  }
  if (n - i == 3) {
    compute(s0, grp_of(i));
    load(s0, grp_of(i + 2));
    compute(s1, grp_of(i + 1));
    compute(s0, grp_of(i + 2));
  } else {
    compute(s0, grp_of(i));
    if (n - i == 2) compute(s1, grp_of(i + 1));
  }
  if constexpr (PARTIALS) return;

  // Partial sums: red[wk][wn][(b, nt, v)][lane]
  constexpr int KK = kept(WK);
  constexpr int REGS = RB * NT * 4;
  auto slot = [&](int k) { return red + static_cast<size_t>(k * WN + wn) * REGS * 64 + lane; };
  auto put = [&](float* dst) {
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int v = 0; v < 4; ++v) dst[((b * NT + nt) * 4 + v) * 64] = acc[b][nt][v];
  };
  if constexpr (KK < WK) {
    if (wk >= KK) put(slot(wk - KK));
    __syncthreads();
    if (wk < KK) {
      const float* src = slot(wk);
#pragma unroll
      for (int b = 0; b < RB; ++b)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
          for (int v = 0; v < 4; ++v) acc[b][nt][v] = acc[b][nt][v] + src[((b * NT + nt) * 4 + v) * 64];
      put(slot(wk));   // the wave overwrites only what it has just read
    }
  } else {
    put(slot(wk));
  }
  __syncthreads();
  // Four consecutive columns per thread, NT * WN tiles of a row side by side.
  constexpr int CH = 4 * NT * WN;   // 4-column chunks per row
  for (int e = threadIdx.x; e < 16 * RB * CH; e += WK * WN * 64) {
    const int ch = e % CH, row = e / CH;
    const int wc = ch / (4 * NT), nt = (ch / 4) % NT, cq = ch & 3;
    const int m = rt * RB * 16 + row;
    const int tile = tile0 + wc * NT + nt;
    if (m >= M || tile >= ntiles) continue;
    const int b = row >> 4, jj = (row >> 2) & 3, v = row & 3;
    const float* src = red + (static_cast<size_t>(wc) * REGS + (b * NT + nt) * 4 + v) * 64 + jj * 16 + cq * 4;
    float4 s = *reinterpret_cast<const float4*>(src);
#pragma unroll
    for (int k = 1; k < KK; ++k) {
      const float4 o = *reinterpret_cast<const float4*>(src + static_cast<size_t>(k) * WN * REGS * 64);
      s.x += o.x;
      s.y += o.y;
      s.z += o.z;
      s.w += o.w;
    }
    const float xs = mb.xs[m];
    const int col = tile * 16 + cq * 4;
    const float f0 = epilogue(s.x, xs, mb.bias, bias_dtype, col), f1 = epilogue(s.y, xs, mb.bias, bias_dtype, col + 1);
    const float f2 = epilogue(s.z, xs, mb.bias, bias_dtype, col + 2), f3 = epilogue(s.w, xs, mb.bias, bias_dtype, col + 3);
    const int64_t o = static_cast<int64_t>(m) * N + col;
    if (y_dtype == PQ_F32) {
      *reinterpret_cast<float4*>(static_cast<float*>(mb.y) + o) = make_float4(f0, f1, f2, f3);
    } else if (y_dtype == PQ_F16) {
      *reinterpret_cast<uint2*>(static_cast<uint16_t*>(mb.y) + o) = make_uint2(pk_f16(f0, f1), pk_f16(f2, f3));
    } else {
      *reinterpret_cast<uint2*>(static_cast<uint16_t*>(mb.y) + o) =
          make_uint2(pq_f32_to_bf16(f0) | (static_cast<uint32_t>(pq_f32_to_bf16(f1)) << 16),
                     pq_f32_to_bf16(f2) | (static_cast<uint32_t>(pq_f32_to_bf16(f3)) << 16));
    }
  }
}

template <int RB, int NT, int WK, int WN, bool NTW, bool PARTIALS>
void launch_mid_t(pq::GemmGroup grp, int bias_dtype, int y_dtype, int M, int K, hipStream_t stream) {
  grp.first[0] = 0;
  for (int i = 0; i < grp.count; ++i) grp.first[i + 1] = grp.first[i] + (grp.mem[i].n / 16 + NT * WN - 1) / (NT * WN);
  const int nrt = ((M + 15) / 16 + RB - 1) / RB;
  const unsigned grid = static_cast<unsigned>(grp.first[grp.count]) * static_cast<unsigned>(nrt);
  const size_t lds = PARTIALS ? 0 : lds_bytes<RB, NT, WK, WN>();
  gemm_mid<RB, NT, WK, WN, NTW, PARTIALS><<<grid, WK * WN * 64, lds, stream>>>(grp, bias_dtype, y_dtype, M, K);
}

}  // namespace pqmid
