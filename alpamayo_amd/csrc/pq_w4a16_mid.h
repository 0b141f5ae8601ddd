// W4A16 GEMM for 17 to a few hundred rows, on tiled fp16 activations: the
// structure of the W4A8 one (pq_gemm_mid.h) -- a wave owns RB x NT blocks of
// 16 x 16 outputs and one of WK parts of K, operands straight into registers
// two groups ahead, no barrier before the final LDS sum -- with the weights
// dequantized once per wave and block and v_mfma_f32_16x16x32_f16 summing over
// the groups (no scaling per group).  The dequantization, 56 VALU
// instructions per 16 columns and group, is what RB rows blocks share.
//
// A row's outputs are the same bits in every configuration, so that a group of
// linears returns what its members return alone: part p of K is every
// kParts16-th group from group p on, a wave walks one part or two, every part's
// sum starts from zero and goes to LDS, and there the parts are added in one
// order.  (Contiguous parts, as in the W4A8 kernel, keep a workgroup's waves
// further apart in A and took 1 to 4 % longer on a decoder layer's linears.)
#pragma once

#include "pq_gemm_mid.h"
#include "pq_w4a16.h"

namespace pqmid {

using namespace pqw16;

constexpr int kParts16 = 8;

template <int RB, int NT, int WN>
constexpr size_t lds_bytes16() { return static_cast<size_t>(kParts16) * WN * RB * NT * 4 * 64 * sizeof(float); }

// Steps 0 .. n - 1 (n >= 1) of load and compute on two register stages, loads
// two steps ahead; the tail is peeled so that no load sits behind a branch
// (the compiler would wait for every load at the join).
template <typename S, typename L, typename C>
__device__ __forceinline__ void walk(int n, const L& load, const C& compute) {
  S s0, s1;
  load(s0, 0);
  load(s1, min(1, n - 1));
  int i = 0;
  for (; i + 3 < n; i += 2) {
    compute(s0);
    load(s0, i + 2);
    compute(s1);
    load(s1, i + 3);
  }
  if (n - i == 3) {
    compute(s0);
    load(s0, i + 2);
    compute(s1);
    compute(s0);
  } else {
    compute(s0);
    if (n - i == 2) compute(s1);
  }
}

template <int RB, int NT>
struct Stage16 {
  v8h a[RB][4];
  v4i w[NT];
  uint32_t meta[NT];
};

// (bounds of the 4-wave instance: three workgroups per CU)
// FEW: fewer than two groups of K in some parts (K < 2048), where walk would load a lone group twice and a wave's second
// part would start with nothing in flight: N = 4096, K = 1024, M = 400 21.9 -> 17.9 us with the rotation, K = 1536 23.9 ->
// 22.7.  An instance of its own, because the branch costs the larger ones registers (4 x 2 blocks 5 % at K = 4096).
template <int RB, int NT, int WK, int WN, bool FEW>
__global__ __launch_bounds__(WK * WN * 64, WK * WN == 4 ? 3 : 2) void w16_mid(const W16Group grp, int bias_dtype, int y_dtype, int M, int K) {
  extern __shared__ __attribute__((aligned(16))) float red[];
  const int G = K >> 7;
  const int nrb = (M + 15) >> 4;
  const int nrt = (nrb + RB - 1) / RB;
  // each XCD a contiguous run of (column unit, row tile) pairs, row tiles innermost
  const int q8 = gridDim.x >> 3, r8 = gridDim.x & 7, xcd = blockIdx.x & 7;
  const int t = xcd * q8 + min(xcd, r8) + (blockIdx.x >> 3);
  const int unit = t / nrt, rt = t - unit * nrt;
  int mi = 0;
#pragma unroll
  for (int i = 1; i < pq::kMaxGroup; ++i)
    if (i < grp.count && unit >= grp.first[i]) mi = i;
  const W16Args& mb = grp.mem[mi];
  const int N = mb.n;
  const int ntiles = N >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wk = wave / WN, wn = wave % WN;
  const int lane = threadIdx.x & 63;
  const int c = lane & 15, j = lane >> 4;
  const int tile0 = (unit - grp.first[mi]) * (NT * WN);

  // Tiles past N and row blocks past M are clamped; their results are not stored.
  const uint8_t* wp[NT];
  const uint32_t* mp[NT];
  const uint8_t* ap[RB];
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
    ap[b] = reinterpret_cast<const uint8_t*>(mb.x) + static_cast<int64_t>(rb) * G * 4096;
    ar[b] = min(M - rb * 16, 16);
    al[b] = (j * ar[b] + min(static_cast<uint32_t>(c), ar[b] - 1)) * 16;   // rows past M repeat the last
  }
  const uint32_t l16 = lane * 16, c4 = c * 4;
  auto load = [&](Stage16<RB, NT>& s, int g) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      s.w[nt] = *reinterpret_cast<const v4i*>(scalar_base<true>(wp[nt] + g * 1024) + l16);
      s.meta[nt] = *reinterpret_cast<const uint32_t*>(scalar_base<true>(mp[nt] + g * 16) + c4);
    }
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        s.a[b][q] = *reinterpret_cast<const v8h*>(scalar_base<true>(ap[b] + (4 * g + q) * 64 * ar[b]) + al[b]);
  };

  v4f acc[RB][NT];
  auto compute = [&](const Stage16<RB, NT>& s) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const v2h s2 = meta_s2(s.meta[nt]), z2 = meta_z2(s.meta[nt]);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const v8h wv = dequant8(static_cast<uint32_t>(s.w[nt][q]), s2, z2);
#pragma unroll
        for (int b = 0; b < RB; ++b) acc[b][nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(s.a[b][q], wv, acc[b][nt], 0, 0, 0);
      }
    }
  };

  // The sums of parts: red[part][wn][(b, nt, v)][lane]
  constexpr int REGS = RB * NT * 4;
  auto put = [&](int part) {
    float* dst = red + static_cast<size_t>(part * WN + wn) * REGS * 64 + lane;
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int v = 0; v < 4; ++v) dst[((b * NT + nt) * 4 + v) * 64] = acc[b][nt][v];
  };
  auto zero = [&] {
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[b][nt] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  };
  // Wave wk walks parts wk, wk + WK, .. one after the other (the host keeps kParts16 <= G).  One loop over both of a
  // 4-wave instance, with the sum put away in its middle, costs it its third wave per SIMD.
  if constexpr (!FEW) {
#pragma unroll 1
    for (int part = wk; part < kParts16; part += WK) {
      zero();
      walk<Stage16<RB, NT>>((G - part + kParts16 - 1) / kParts16,
                            [&](Stage16<RB, NT>& s, int i) { load(s, part + i * kParts16); }, compute);
      put(part);
    }
  } else if (2 * WK == kParts16 && G == kParts16) {   // one group a part: both parts' loads first
    Stage16<RB, NT> s0, s1;
    load(s0, wk);
    load(s1, wk + WK);
    zero();
    compute(s0);
    put(wk);
    zero();
    compute(s1);
    put(wk + WK);
  } else {
#pragma unroll 1
    for (int part = wk; part < kParts16; part += WK) {
      Stage16<RB, NT> s0, s1;
      load(s0, part);
      zero();
      if (part + kParts16 < G) {
        load(s1, part + kParts16);
        compute(s0);
        compute(s1);
      } else {
        compute(s0);
      }
      put(part);
    }
  }
  __syncthreads();
  constexpr int CH = 4 * NT * WN;   // 4-column chunks per row
  for (int e = threadIdx.x; e < 16 * RB * CH; e += WK * WN * 64) {
    const int ch = e % CH, row = e / CH;
    const int wc = ch / (4 * NT), nt = (ch / 4) % NT, cq = ch & 3;
    const int m = rt * RB * 16 + row;
    const int tile = tile0 + wc * NT + nt;
    if (m >= M || tile >= ntiles) continue;
    const int b = row >> 4, jj = (row >> 2) & 3, v = row & 3;
    const float* src = red + (static_cast<size_t>(wc) * REGS + (b * NT + nt) * 4 + v) * 64 + jj * 16 + cq * 4;
    float4 p[kParts16];
#pragma unroll
    for (int k = 0; k < kParts16; ++k)
      p[k] = *reinterpret_cast<const float4*>(src + static_cast<size_t>(k) * WN * REGS * 64);
#pragma unroll
    for (int d = 1; d < kParts16; d *= 2)   // neighbours first
#pragma unroll
      for (int k = 0; k < kParts16; k += 2 * d) {
        p[k].x += p[k + d].x;
        p[k].y += p[k + d].y;
        p[k].z += p[k + d].z;
        p[k].w += p[k + d].w;
      }
    float f[4] = {p[0].x, p[0].y, p[0].z, p[0].w};
    const int col = tile * 16 + cq * 4;
    if (mb.bias != nullptr) {
#pragma unroll
      for (int q = 0; q < 4; ++q) f[q] = f[q] + pq_load_dyn(mb.bias, bias_dtype, col + q);
    }
    const int64_t o = static_cast<int64_t>(m) * N + col;
    if (y_dtype == PQ_F32) {
      *reinterpret_cast<float4*>(static_cast<float*>(mb.y) + o) = make_float4(f[0], f[1], f[2], f[3]);
    } else if (y_dtype == PQ_F16) {
      *reinterpret_cast<uint2*>(static_cast<uint16_t*>(mb.y) + o) = make_uint2(pk_f16(f[0], f[1]), pk_f16(f[2], f[3]));
    } else {
      *reinterpret_cast<uint2*>(static_cast<uint16_t*>(mb.y) + o) =
          make_uint2(pq_f32_to_bf16(f[0]) | (static_cast<uint32_t>(pq_f32_to_bf16(f[1])) << 16),
                     pq_f32_to_bf16(f[2]) | (static_cast<uint32_t>(pq_f32_to_bf16(f[3])) << 16));
    }
  }
}

template <int RB, int NT, int WK, int WN>
void launch_w16_mid_t(W16Group grp, int bias_dtype, int y_dtype, int M, int K, hipStream_t stream) {
  grp.first[0] = 0;
  for (int i = 0; i < grp.count; ++i) grp.first[i + 1] = grp.first[i] + (grp.mem[i].n / 16 + NT * WN - 1) / (NT * WN);
  const int nrt = ((M + 15) / 16 + RB - 1) / RB;
  const unsigned grid = static_cast<unsigned>(grp.first[grp.count]) * static_cast<unsigned>(nrt);
  const size_t lds = lds_bytes16<RB, NT, WN>();
  if (K < 2 * kParts16 * 128)
    w16_mid<RB, NT, WK, WN, true><<<grid, WK * WN * 64, lds, stream>>>(grp, bias_dtype, y_dtype, M, K);
  else
    w16_mid<RB, NT, WK, WN, false><<<grid, WK * WN * 64, lds, stream>>>(grp, bias_dtype, y_dtype, M, K);
}

}  // namespace pqmid
