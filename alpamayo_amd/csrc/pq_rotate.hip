// Stage 1 and 2 of the W4A8 linear on gfx950:
//   pq_rotate           -- the rotation::rotate op (pairwise Givens + channel scale)
//   pq_rotate_quant_i8  -- rotation + per-token absmax + int8 quant, one pass
//   pq_quant_i8         -- per-token int8 quant of an existing tensor
//
// Reference semantics: kernels/paroquant_kernels/src/rotation.cuh:247-337
// (scale-multiply, KROT Givens layers xi' = c xi + s xj, xj' = -s xi + c xj
// on group-local pair indices, fp32 math, result rounded to the storage
// dtype) and vLLM's dynamic per-token int8 quant (scale = absmax/127,
// q = rne(x * 127/absmax)) as called at
// src/alpamayo_r1/utils/quantization/paroquant_marlin_w4a8.py:319-333.
//
// All updates are written with explicit fmaf and the file is compiled with
// -ffp-contract=off, so the float32 sequence is fixed:
//   xi' = fma(xi, c, xj*s),  xj' = fma(xj, c, -(xi*s)).
#include <algorithm>
#include <type_traits>

#include "pq_chain.h"
#include "pq_device.h"
#include "pq_internal.h"

using pqd::quant4;

namespace {

constexpr int kRotRows = 16;   // rows per workgroup of the plain rotation kernel


// ---------------------------------------------------------------------------
// rotation::rotate.  A workgroup of 4 waves takes 16 rows x 128 channels (for
// group 64 the chunk holds two groups).  The 64 pairs' indices (masked to the
// group, so a bad index can never address outside the tile) and cos/sin of
// every layer are derived once per workgroup into LDS -- each sincos serves
// 16 rows.  Wave w owns rows 4w .. 4w+3 as a channel-major LDS tile (one
// float4 = the wave's 4 rows of a channel), so lane l applies a layer to its
// pair with two 16-byte reads and two 16-byte writes.
// ---------------------------------------------------------------------------
//
// MX: instead of the rotated values, their OCP MXFP4 quantization (fused
// rotate + quant): y receives the E2M1 codes [rows][h/2] (element 2i in the
// low nibble of byte i) and sc the E8M0 scales [rows][h/32] (0xFF when the
// block holds a NaN).  Lane l quantizes channels 2l, 2l+1 of its wave's rows;
// the 16 lanes of a 32-channel block exchange their absmax by shuffles.
constexpr int kRotWaves = 4;
constexpr int kRotRowsPerWave = 4;
constexpr int kRotMaxLayers = 16;

template <int DT, int G, bool SCALE, bool MX>
__global__ __launch_bounds__(kRotWaves * 64) void rotate_kernel(const void* __restrict__ x, void* __restrict__ y,
                                                                uint8_t* __restrict__ sc,
                                                                const int16_t* __restrict__ idx,
                                                                const void* __restrict__ theta,
                                                                const void* __restrict__ scales, int64_t rows,
                                                                int h, int krot) {
  static_assert(kRotRows == kRotWaves * kRotRowsPerWave && kRotRowsPerWave == 4, "a float4 per channel and wave");
  __shared__ float4 tile[kRotWaves][128];
  __shared__ float2 s_cs[kRotMaxLayers][64];
  __shared__ uint32_t s_ij[kRotMaxLayers][64];
  constexpr int NT = kRotWaves * 64;
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int w = t >> 6;
  const int64_t row0 = static_cast<int64_t>(blockIdx.x) * kRotRows;
  const int ch0 = blockIdx.y * 128;

  // Layer parameters of the chunk's 64 pairs.  A pair past h (the second
  // half of a 64-channel tail) turns its own two channels, which hold zeros
  // and are never stored, by the identity.
  for (int e = t; e < krot * 64; e += NT) {
    const int r = e >> 6, p = e & 63;
    const int P = blockIdx.y * 64 + p;   // pair index within the row; theta column
    float c = 1.0f, sn = 0.0f;
    uint32_t ij = static_cast<uint32_t>(2 * p) | (static_cast<uint32_t>(2 * p + 1) << 8);
    if (P < (h >> 1)) {
      const int gi = P / (G / 2);
      const int pp = P % (G / 2);
      const int base = gi * G - ch0;   // group start inside the 128-channel tile
      const int64_t o = static_cast<int64_t>(r) * h + gi * G + 2 * pp;
      const int i = base + (idx[o] & (G - 1));
      const int j = base + (idx[o + 1] & (G - 1));
      const float th = pq_load_as_f32<DT>(theta, static_cast<int64_t>(r) * (h >> 1) + P);
      // cos and sin of the stored angle in float64, rounded once to float32:
      // the values the host derives for the fused kernels' operands, so this
      // kernel and those agree bit for bit
      double sd, cd;
      sincos(static_cast<double>(th), &sd, &cd);
      c = static_cast<float>(cd);
      sn = static_cast<float>(sd);
      ij = static_cast<uint32_t>(i) | (static_cast<uint32_t>(j) << 8);
    }
    s_cs[r][p] = make_float2(c, sn);
    s_ij[r][p] = ij;
  }
  // Wave w loads its own rows: lane l channels 2l, 2l+1 of each (coalesced).
  float4* wt = tile[w];
  {
    const int ch = ch0 + 2 * lane;
    float s0 = 1.0f, s1 = 1.0f;
    if (SCALE && ch < h) {
      s0 = pq_load_as_f32<DT>(scales, ch);
      s1 = pq_load_as_f32<DT>(scales, ch + 1);
    }
    float va[kRotRowsPerWave], vb[kRotRowsPerWave];
#pragma unroll
    for (int rr = 0; rr < kRotRowsPerWave; ++rr) {
      const int64_t row = row0 + w * kRotRowsPerWave + rr;
      va[rr] = 0.0f;
      vb[rr] = 0.0f;
      if (row < rows && ch < h) {
        va[rr] = pq_load_as_f32<DT>(x, row * h + ch);
        vb[rr] = pq_load_as_f32<DT>(x, row * h + ch + 1);
        if (SCALE) {
          va[rr] = va[rr] * s0;
          vb[rr] = vb[rr] * s1;
        }
      }
    }
    wt[2 * lane] = make_float4(va[0], va[1], va[2], va[3]);
    wt[2 * lane + 1] = make_float4(vb[0], vb[1], vb[2], vb[3]);
  }
  __syncthreads();

  for (int r = 0; r < krot; ++r) {
    const float2 cs = s_cs[r][lane];
    const uint32_t ij = s_ij[r][lane];
    const int i = static_cast<int>(ij & 0xffu), j = static_cast<int>(ij >> 8);
    const float4 xi = wt[i];
    const float4 xj = wt[j];
    float4 ni, nj;
    ni.x = fmaf(xi.x, cs.x, xj.x * cs.y);
    nj.x = fmaf(xj.x, cs.x, -(xi.x * cs.y));
    ni.y = fmaf(xi.y, cs.x, xj.y * cs.y);
    nj.y = fmaf(xj.y, cs.x, -(xi.y * cs.y));
    ni.z = fmaf(xi.z, cs.x, xj.z * cs.y);
    nj.z = fmaf(xj.z, cs.x, -(xi.z * cs.y));
    ni.w = fmaf(xi.w, cs.x, xj.w * cs.y);
    nj.w = fmaf(xj.w, cs.x, -(xi.w * cs.y));
    wt[i] = ni;
    wt[j] = nj;
    // The sub-tile is this wave's alone, and a wave's LDS operations complete
    // in issue order: the next layer's reads see these writes without a
    // workgroup barrier.  The fence keeps the compiler from moving them.
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
  }

  // Lane l of wave w holds channels 2l, 2l+1 of the wave's 4 rows.
  const float4 fa = wt[2 * lane], fb = wt[2 * lane + 1];
  const float va[kRotRowsPerWave] = {fa.x, fa.y, fa.z, fa.w};
  const float vb[kRotRowsPerWave] = {fb.x, fb.y, fb.z, fb.w};
  const int ch = ch0 + 2 * lane;
  if constexpr (MX) {
    // a 32-channel block = 16 lanes: absmax and the NaN flag over them by shuffles
#pragma unroll
    for (int rr = 0; rr < kRotRowsPerWave; ++rr) {
      float am = fmaxf(fabsf(va[rr]), fabsf(vb[rr]));
      int nn = (va[rr] != va[rr]) || (vb[rr] != vb[rr]) ? 1 : 0;
#pragma unroll
      for (int d = 1; d < 16; d <<= 1) {
        am = fmaxf(am, __shfl_xor(am, d));
        nn |= __shfl_xor(nn, d);
      }
      const int ex = pqd::mx_shared_exp(am);
      const float inv = pqd::mx_inv_scale(ex);
      const uint32_t code = pqd::mx_e2m1(va[rr] * inv) | (pqd::mx_e2m1(vb[rr] * inv) << 4);
      const int64_t row = row0 + w * kRotRowsPerWave + rr;
      if (row < rows && ch < h) {
        static_cast<uint8_t*>(y)[row * (h >> 1) + (ch >> 1)] = static_cast<uint8_t>(code);
        if ((lane & 15) == 0) sc[row * (h >> 5) + (ch >> 5)] = nn ? 0xFFu : static_cast<uint8_t>(ex + 127);
      }
    }
  } else {
#pragma unroll
    for (int rr = 0; rr < kRotRowsPerWave; ++rr) {
      const int64_t row = row0 + w * kRotRowsPerWave + rr;
      if (row < rows && ch < h) {
        pq_store_from_f32<DT>(y, row * h + ch, va[rr]);
        pq_store_from_f32<DT>(y, row * h + ch + 1, vb[rr]);
      }
    }
  }
}

template <int NT>
__device__ __forceinline__ float block_max(float v, float* red) {
  constexpr int NW = NT / 64;
  v = pq_wave_max_nonneg(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float m = red[0];
#pragma unroll
  for (int k = 1; k < NW; ++k) m = fmaxf(m, red[k]);
  return m;
}

template <int DT>
__device__ __forceinline__ void load8(const void* base, int64_t elem, float f[8]) {
  if constexpr (DT == PQ_F32) {
    const float4* p = reinterpret_cast<const float4*>(static_cast<const float*>(base) + elem);
    const float4 a = p[0], b = p[1];
    f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w;
    f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
  } else {
    const uint4 u = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(base) + elem);
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint16_t lo = static_cast<uint16_t>(w[e] & 0xffffu), hi = static_cast<uint16_t>(w[e] >> 16);
      if constexpr (DT == PQ_F16) {
        f[2 * e] = pq_f16_to_f32(lo);
        f[2 * e + 1] = pq_f16_to_f32(hi);
      } else {
        f[2 * e] = pq_bf16_to_f32(lo);
        f[2 * e + 1] = pq_bf16_to_f32(hi);
      }
    }
  }
}



// ---------------------------------------------------------------------------
// Split rotation for decode-size inputs: one wave per 128-channel group and
// MR rows (M <= MR <= 16; rows past M repeat row M-1 and are not stored), so
// the K/128 groups run on K/128 waves spread over the chip and every
// parameter byte is read once.  Writes the rotated rows (fp16 when
// materialized in fp16, else fp32) and each row's absmax per group; the
// GEMM that follows derives the token scale and quantizes.  One wave per
// workgroup: the waves share nothing, and single-wave workgroups spread over
// more CUs sooner (decode layer at M = 1: 43.5 -> 42.0 us against four waves
// per workgroup, 42.4 us with two).
// ---------------------------------------------------------------------------
constexpr int kSplitWaves = 1;

// With the RMSNorm prologue and one row per wave, WPB = kSplitNormWaves
// waves per workgroup take WPB consecutive groups of the row and share its
// sum of squares: wave w sums the chunk classes w, w + WPB, ... of the row,
// the eight partials meet in LDS and every wave adds them in the fixed order,
// which gives the bits a single wave gets summing the whole row, with 1/WPB
// of the loads per wave.  Four waves: against one wave per workgroup summing
// the whole row, the 36-layer verify block (M = 16) 2.160 -> 2.120 ms and the
// fused decode chain (M = 1) 1.550 -> 1.533 ms; eight waves 2.130 / 1.552 ms
// (fewer CUs at M = 1), two 2.128 / 1.533 ms.
constexpr int kSplitNormWaves = 4;

template <int DT, int KP, bool MAT16, int MR, bool NORM, int WPB = kSplitWaves>
__global__ __launch_bounds__(WPB * 64) void rotate_split_kernel(const void* __restrict__ x, const pq::RotGroup grp,
                                                                int M, int h, int krot, unsigned flags,
                                                                const pq::NormArgs nm) {
  constexpr bool kCoop = WPB > 1;
  static_assert(WPB == 1 || (pqd::kSumClasses % WPB == 0 && MR == 1 && NORM),
                "shared row sums: one row per wave, RMSNorm prologue");
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int g = blockIdx.x * WPB + wv;
  const pq::RotMember& mb = grp.mem[blockIdx.y];
  // the normalized rows and the residual sum are the same for every member: member 0 writes them
  const bool first = blockIdx.y == 0;
  // grid.z: chunks of MR rows; the row pointers move to the chunk's first row
  const int row0 = blockIdx.z * MR;
  const int64_t e0 = static_cast<int64_t>(row0) * h;
  constexpr int xsz = DT == PQ_F32 ? 4 : 2;
  auto at = [](const void* p, int64_t bytes) -> void* {
    return p == nullptr ? nullptr : const_cast<char*>(static_cast<const char*>(p)) + bytes;
  };
  float rinv = -1.0f;
  if constexpr (kCoop) {
    if (nm.mode == PQ_PRO_RMSNORM) {   // uniform over the launch
      constexpr int NC = pqd::kSumClasses / WPB;
      __shared__ float s_part[pqd::kSumClasses][64];
      float pw[NC];
      pqd::row_sumsq_part<DT, NC, NC >= 4 ? 1 : 4 / NC>(at(x, e0 * xsz), at(nm.res, e0 * xsz), 0, h, lane, wv, WPB,
                                                         pw);
#pragma unroll
      for (int j = 0; j < NC; ++j) s_part[wv + j * WPB][lane] = pw[j];
      pqd::lds_barrier();
      float p[pqd::kSumClasses];
#pragma unroll
      for (int c = 0; c < pqd::kSumClasses; ++c) p[c] = s_part[c][lane];
      rinv = pqd::rms_inv(pqd::row_sumsq_total(p), h, nm.eps);
    }
  }
  if (g >= (h >> 7)) return;   // whole waves, after the workgroup's only barrier
  pqd::rotate_group_rows<DT, KP, MAT16, MR, NORM>(
      at(x, e0 * xsz), mb.rot_idx, mb.rot_cs, mb.scales, at(mb.out, e0 * (MAT16 ? 2 : 4)),
      mb.out_scale + static_cast<int64_t>(row0) * (h >> 7), min(MR, M - row0), h, krot, flags, g, lane,
      at(nm.res, e0 * xsz), nm.w, first ? at(nm.h_out, e0 * xsz) : nullptr, first ? at(nm.s_out, e0 * xsz) : nullptr,
      nm.eps, nm.mode, rinv);
}

// Per-token int8 quantization of the split rotation's rows, for token counts
// where the GEMM should not re-derive it in every workgroup.  grid (chunks of
// 2048 channels, rows, members); each thread quantizes 8 channels.  The token
// absmax is the largest group maximum in the unsigned order of its bits (the
// maxima are >= 0), as the rotated decode GEMM takes it, so both give the
// same codes and scales.
template <bool MAT16>
__global__ __launch_bounds__(256) void quant_split_kernel(const pq::QuantGroup grp, int h) {
  const pq::QuantMember& mb = grp.mem[blockIdx.z];
  const int row = blockIdx.y;
  const int G = h >> 7;
  const int lane = threadIdx.x & 63;
  const int c8 = (blockIdx.x * 256 + threadIdx.x) * 8;
  // the thread's 8 values are requested together with the group maxima (one
  // memory round trip, not two); threads past h re-read the row's last 8
  const int64_t o = static_cast<int64_t>(row) * h + min(c8, h - 8);
  uint4 v16;
  float4 va, vb;
  if constexpr (MAT16) {
    v16 = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(mb.xr) + o);
  } else {
    va = *reinterpret_cast<const float4*>(static_cast<const float*>(mb.xr) + o);
    vb = *reinterpret_cast<const float4*>(static_cast<const float*>(mb.xr) + o + 4);
  }
  const float* gm = mb.gmax + static_cast<int64_t>(row) * G;
  uint32_t u = 0;
  // Up to 128 groups (k <= 16384 on every caller): two maxima per lane,
  // requested together, with clamped indices (a repeated maximum changes
  // nothing); a loop over them waited for each before requesting the next.
  if (G <= 128) {
    u = max(__float_as_uint(gm[min(lane, G - 1)]), __float_as_uint(gm[min(lane + 64, G - 1)]));
  } else {
    for (int i = lane; i < G; i += 64) u = max(u, __float_as_uint(gm[i]));
  }
  const float am = __uint_as_float(pq_wave_umax(u));
  if (c8 >= h) return;
  const float inv = pqd::inv_scale(am);
  uint2 q;
  if constexpr (MAT16) {
    q.x = pqd::quant4_f16(v16.x, v16.y, inv);
    q.y = pqd::quant4_f16(v16.z, v16.w, inv);
  } else {
    q.x = pqd::quant4(va.x, va.y, va.z, va.w, inv);
    q.y = pqd::quant4(vb.x, vb.y, vb.z, vb.w, inv);
  }
  *reinterpret_cast<uint2*>(mb.xq + (grp.tiled ? pqd::a_tile_offset(row, c8, grp.tiled, G) : o)) = q;
  if (c8 == 0) mb.xscale[row] = am / 127.0f;
}

template <int DT, int KP, bool MAT16, bool NORM>
void launch_split_kp(const void* x, const pq::RotGroup& grp, int M, int h, int krot, unsigned flags,
                     const pq::NormArgs& nm, int rows_per_wave, hipStream_t stream) {
  const int rows = rows_per_wave > 0 && rows_per_wave < M ? rows_per_wave : M;
  if constexpr (NORM) {
    if (rows == 1 && nm.mode == PQ_PRO_RMSNORM) {
      constexpr int W = kSplitNormWaves;
      const dim3 grid(static_cast<unsigned>((h / 128 + W - 1) / W), static_cast<unsigned>(grp.count),
                      static_cast<unsigned>(M));
      rotate_split_kernel<DT, KP, MAT16, 1, true, W><<<grid, W * 64, 0, stream>>>(x, grp, M, h, krot, flags, nm);
      return;
    }
  }
  const dim3 grid(static_cast<unsigned>((h / 128 + kSplitWaves - 1) / kSplitWaves), static_cast<unsigned>(grp.count),
                  static_cast<unsigned>((M + rows - 1) / rows));
#define PQ_SPLIT(MR_)                                                                                      \
  if (rows <= MR_) {                                                                                       \
    rotate_split_kernel<DT, KP, MAT16, MR_, NORM><<<grid, kSplitWaves * 64, 0, stream>>>(x, grp, M, h, krot, \
                                                                                        flags, nm);          \
    return;                                                                                                \
  }
  PQ_SPLIT(1) PQ_SPLIT(2) PQ_SPLIT(4) PQ_SPLIT(8) PQ_SPLIT(16)
#undef PQ_SPLIT
}

template <int DT, bool NORM>
void launch_split_norm(const void* x, const pq::RotGroup& grp, int M, int h, int krot, unsigned flags,
                       const pq::NormArgs& nm, int rpw, hipStream_t stream) {
  const bool mat16 = (flags & PQ_RQ_MATERIALIZE_FP16) != 0;
  if (krot <= 8) {
    if (mat16) launch_split_kp<DT, 8, true, NORM>(x, grp, M, h, krot, flags, nm, rpw, stream);
    else launch_split_kp<DT, 8, false, NORM>(x, grp, M, h, krot, flags, nm, rpw, stream);
  } else {
    if (mat16) launch_split_kp<DT, 16, true, NORM>(x, grp, M, h, krot, flags, nm, rpw, stream);
    else launch_split_kp<DT, 16, false, NORM>(x, grp, M, h, krot, flags, nm, rpw, stream);
  }
}

template <int DT>
void launch_split_dt(const void* x, const pq::RotGroup& grp, int M, int h, int krot, unsigned flags,
                     const pq::NormArgs* norm, int rpw, hipStream_t stream) {
  if (norm != nullptr) launch_split_norm<DT, true>(x, grp, M, h, krot, flags, *norm, rpw, stream);
  else launch_split_norm<DT, false>(x, grp, M, h, krot, flags, pq::NormArgs{}, rpw, stream);
}

// Per-token quant of an existing activation: absmax pass, then quant pass.
template <int DT, int NT>
__global__ __launch_bounds__(NT) void quant_kernel(const void* __restrict__ x, int8_t* __restrict__ xq,
                                                   float* __restrict__ xscale, int64_t rows, int h) {
  __shared__ float red[NT / 64];
  const int t = threadIdx.x;
  for (int64_t row = blockIdx.x; row < rows; row += gridDim.x) {
    const int64_t rbase = row * h;
    float amax = 0.0f;
    for (int v = t; v < (h >> 3); v += NT) {
      float f[8];
      load8<DT>(x, rbase + 8 * v, f);
#pragma unroll
      for (int e = 0; e < 8; ++e) amax = fmaxf(amax, fabsf(f[e]));
    }
    const float am = block_max<NT>(amax, red);
    const float inv = pqd::inv_scale(am);
    if (t == 0) xscale[row] = am / 127.0f;
    for (int v = t; v < (h >> 3); v += NT) {
      float f[8];
      load8<DT>(x, rbase + 8 * v, f);
      uint2 o;
      o.x = quant4(f[0], f[1], f[2], f[3], inv);
      o.y = quant4(f[4], f[5], f[6], f[7], inv);
      *reinterpret_cast<uint2*>(xq + rbase + 8 * v) = o;
    }
    __syncthreads();
  }
}

template <int DT, int G, bool SCALE>
void launch_rotate(const void* x, void* y, uint8_t* sc, const int16_t* idx, const void* theta, const void* scales,
                   int64_t rows, int h, int krot, hipStream_t stream) {
  dim3 grid(static_cast<unsigned>((rows + kRotRows - 1) / kRotRows), static_cast<unsigned>((h + 127) / 128));
  if (sc != nullptr)
    rotate_kernel<DT, G, SCALE, true><<<grid, kRotWaves * 64, 0, stream>>>(x, y, sc, idx, theta, scales, rows, h, krot);
  else
    rotate_kernel<DT, G, SCALE, false><<<grid, kRotWaves * 64, 0, stream>>>(x, y, sc, idx, theta, scales, rows, h,
                                                                            krot);
}

// The register chain (pq_chain.h) from 4 M elements on: below, a workgroup's
// chain serves too few rows to pay for being derived (fp16, 8 layers, tile
// form -> chain in us: 512 x 4096 9.6 -> 10.0, 1024 x 4096 15.6 -> 12.9, 2100 x
// 4096 27.3 -> 20.1, 1024 x 12288 37.4 -> 25.7; 16 layers 1024 x 4096 24.1 ->
// 18.7; float32, 8 layers, 8192 x 4096 102 -> 58).  One and two layers are
// little to save, from 6 M (1026 x 4096 8.7 -> 9.4, 1465 x 4096 11.8 -> 9.9;
// with MXFP4 codes 11.9 -> 10.3 already).  And 32 rows at least, a step of a
// workgroup: fewer, longer rows derive a chain per 128 channels for them (16 x
// 262144 15.5 -> 22.3, 4 x 1048576 44 -> 72; 33 x 131072 20.1 -> 17.7).
constexpr int64_t kChainElems = 1 << 22, kChainElemsFewLayers = 6000000, kChainRows = 32;

template <int DT, bool MX>
void launch_chain(const void* x, void* y, uint8_t* sc, const int16_t* idx, const void* theta, const void* scales,
                  int64_t rows, int h, int krot, int group, hipStream_t stream) {
  // Slices of the rows for the two workgroups a CU holds, in whole steps of 32 rows.
  const int64_t chunks = (h + 127) / 128;
  const int64_t want = std::max<int64_t>(1, 512 / chunks);
  const int64_t slice = ((rows + want - 1) / want + 31) / 32 * 32;
  const dim3 grid(static_cast<unsigned>((rows + slice - 1) / slice), static_cast<unsigned>(chunks));
#define PQ_CHAIN(K_)                                                                                                 \
  case K_:                                                                                                           \
    pqchain::rotate_chain<DT, K_, MX><<<grid, pqchain::kWaves * 64, 0, stream>>>(x, y, sc, idx, theta, scales, rows, \
                                                                                 h, group, slice);                   \
    break;
  switch (krot) { PQ_CHAIN(1) PQ_CHAIN(2) PQ_CHAIN(4) PQ_CHAIN(8) PQ_CHAIN(16) }
#undef PQ_CHAIN
}

// sc == nullptr: rotated values into y; else MXFP4 codes into y, scales into sc.
template <int DT>
void launch_rotate_dt(const void* x, void* y, uint8_t* sc, const int16_t* idx, const void* theta,
                      const void* scales, int64_t rows, int h, int krot, int group, hipStream_t stream) {
  if (rows >= kChainRows && rows * h >= (krot <= 2 && sc == nullptr ? kChainElemsFewLayers : kChainElems)) {
    if (sc != nullptr) launch_chain<DT, true>(x, y, sc, idx, theta, scales, rows, h, krot, group, stream);
    else launch_chain<DT, false>(x, y, sc, idx, theta, scales, rows, h, krot, group, stream);
    return;
  }
  if (group == 128) {
    if (scales) launch_rotate<DT, 128, true>(x, y, sc, idx, theta, scales, rows, h, krot, stream);
    else launch_rotate<DT, 128, false>(x, y, sc, idx, theta, scales, rows, h, krot, stream);
  } else {
    if (scales) launch_rotate<DT, 64, true>(x, y, sc, idx, theta, scales, rows, h, krot, stream);
    else launch_rotate<DT, 64, false>(x, y, sc, idx, theta, scales, rows, h, krot, stream);
  }
}

constexpr int64_t kMaxGrid = 1 << 20;


template <int DT>
void launch_quant(const void* x, int8_t* xq, float* xscale, int64_t rows, int h, hipStream_t stream) {
  const unsigned grid = static_cast<unsigned>(rows < kMaxGrid ? rows : kMaxGrid);
  quant_kernel<DT, 256><<<grid, 256, 0, stream>>>(x, xq, xscale, rows, h);
}

}  // namespace

namespace pq {
void launch_rotate_split(const void* x, int x_dtype, const RotGroup& grp, int m, int h, int krot, unsigned flags,
                         hipStream_t stream, const NormArgs* norm, int rows_per_wave) {
  switch (x_dtype) {
    case PQ_F32: launch_split_dt<PQ_F32>(x, grp, m, h, krot, flags, norm, rows_per_wave, stream); break;
    case PQ_F16: launch_split_dt<PQ_F16>(x, grp, m, h, krot, flags, norm, rows_per_wave, stream); break;
    default: launch_split_dt<PQ_BF16>(x, grp, m, h, krot, flags, norm, rows_per_wave, stream); break;
  }
}

void launch_quant_split(const QuantGroup& grp, int m, int h, bool mat16, hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>((h / 8 + 255) / 256), static_cast<unsigned>(m), static_cast<unsigned>(grp.count));
  if (mat16) quant_split_kernel<true><<<grid, 256, 0, stream>>>(grp, h);
  else quant_split_kernel<false><<<grid, 256, 0, stream>>>(grp, h);
}

void launch_rotate_quant_group(const void* x, int x_dtype, const RotGroup& grp, int64_t rows, int h, int krot,
                               unsigned flags, hipStream_t stream, const NormArgs* norm) {
  switch (x_dtype) {
    case PQ_F32: launch_rows_f32(x, grp, rows, h, krot, flags, stream, norm); break;
    case PQ_F16: launch_rows_f16(x, grp, rows, h, krot, flags, stream, norm); break;
    default: launch_rows_bf16(x, grp, rows, h, krot, flags, stream, norm); break;
  }
}
}  // namespace pq

extern "C" int pq_rotate(const void* x, void* y, const int16_t* idx_ij, const void* theta, const void* scales,
                         int64_t rows, int64_t h, int krot, int group_size, int dtype, void* stream) {
  PQ_REQUIRE(rows >= 0 && h > 0, PQ_ERR_ARG, "pq_rotate: rows=%lld h=%lld", (long long)rows, (long long)h);
  PQ_REQUIRE(group_size == 64 || group_size == 128, PQ_ERR_UNSUPPORTED,
             "pq_rotate: Unexpected group_size: %d (supported: 64, 128)", group_size);
  PQ_REQUIRE(krot == 1 || krot == 2 || krot == 4 || krot == 8 || krot == 16, PQ_ERR_UNSUPPORTED,
             "pq_rotate: Unsupported KROT = %d; compiled variants: 1/2/4/8/16", krot);
  PQ_REQUIRE(h % group_size == 0, PQ_ERR_ARG, "pq_rotate: h must be divisible by GROUP_SIZE (h=%lld, G=%d)",
             (long long)h, group_size);
  PQ_REQUIRE(h <= (1 << 24), PQ_ERR_ARG, "pq_rotate: h=%lld too large", (long long)h);
  PQ_REQUIRE(dtype == PQ_F32 || dtype == PQ_F16 || dtype == PQ_BF16, PQ_ERR_UNSUPPORTED,
             "pq_rotate: rotate only supports Float, Half, and BFloat16 (dtype code %d)", dtype);
  if (rows == 0) return PQ_OK;
  PQ_REQUIRE(x && y && idx_ij && theta, PQ_ERR_ARG, "pq_rotate: null pointer");
  PQ_REQUIRE((rows + kRotRows - 1) / kRotRows <= 0x7fffffffLL, PQ_ERR_ARG, "pq_rotate: too many rows");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int hh = static_cast<int>(h);
  switch (dtype) {
    case PQ_F32: launch_rotate_dt<PQ_F32>(x, y, nullptr, idx_ij, theta, scales, rows, hh, krot, group_size, s); break;
    case PQ_F16: launch_rotate_dt<PQ_F16>(x, y, nullptr, idx_ij, theta, scales, rows, hh, krot, group_size, s); break;
    default: launch_rotate_dt<PQ_BF16>(x, y, nullptr, idx_ij, theta, scales, rows, hh, krot, group_size, s); break;
  }
  return pq::launch_status("pq_rotate launch");
}

// rotation::rotate followed by OCP MXFP4 quantization of the float32 result,
// in one pass.  The CDNA4 counterpart of the reference's NVFP4
// rotation::rotate_and_quant (kernels/paroquant_kernels/src/rotation.cu:62-111,
// 230-315): the same rotation, a different block format (32-element blocks,
// E8M0 scales, no second-level scale).
extern "C" int pq_rotate_mxfp4(const void* x, uint8_t* q_out, uint8_t* scale_out, const int16_t* idx_ij,
                               const void* theta, const void* scales, int64_t rows, int64_t h, int krot,
                               int group_size, int dtype, void* stream) {
  PQ_REQUIRE(rows >= 0 && h > 0, PQ_ERR_ARG, "pq_rotate_mxfp4: rows=%lld h=%lld", (long long)rows, (long long)h);
  PQ_REQUIRE(group_size == 64 || group_size == 128, PQ_ERR_UNSUPPORTED,
             "pq_rotate_mxfp4: Unexpected group_size: %d (supported: 64, 128)", group_size);
  PQ_REQUIRE(krot == 1 || krot == 2 || krot == 4 || krot == 8 || krot == 16, PQ_ERR_UNSUPPORTED,
             "pq_rotate_mxfp4: Unsupported KROT = %d; compiled variants: 1/2/4/8/16", krot);
  PQ_REQUIRE(h % group_size == 0, PQ_ERR_ARG, "pq_rotate_mxfp4: h must be divisible by GROUP_SIZE (h=%lld, G=%d)",
             (long long)h, group_size);
  PQ_REQUIRE(h <= (1 << 24), PQ_ERR_ARG, "pq_rotate_mxfp4: h=%lld too large", (long long)h);
  PQ_REQUIRE(dtype == PQ_F32 || dtype == PQ_F16 || dtype == PQ_BF16, PQ_ERR_UNSUPPORTED,
             "pq_rotate_mxfp4: dtype code %d (Float, Half or BFloat16)", dtype);
  if (rows == 0) return PQ_OK;
  PQ_REQUIRE(x && q_out && scale_out && idx_ij && theta, PQ_ERR_ARG, "pq_rotate_mxfp4: null pointer");
  PQ_REQUIRE(pq::aligned_to(q_out, 4), PQ_ERR_ARG, "pq_rotate_mxfp4: q_out must be 4-byte aligned");
  PQ_REQUIRE((rows + kRotRows - 1) / kRotRows <= 0x7fffffffLL, PQ_ERR_ARG, "pq_rotate_mxfp4: too many rows");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int hh = static_cast<int>(h);
  switch (dtype) {
    case PQ_F32:
      launch_rotate_dt<PQ_F32>(x, q_out, scale_out, idx_ij, theta, scales, rows, hh, krot, group_size, s);
      break;
    case PQ_F16:
      launch_rotate_dt<PQ_F16>(x, q_out, scale_out, idx_ij, theta, scales, rows, hh, krot, group_size, s);
      break;
    default:
      launch_rotate_dt<PQ_BF16>(x, q_out, scale_out, idx_ij, theta, scales, rows, hh, krot, group_size, s);
      break;
  }
  return pq::launch_status("pq_rotate_mxfp4 launch");
}

// rotation::rotate / rotation::rotate_and_quant_mxfp4 on packed operands
// (pq_rotation_pack): the register-chain rotation of the fused kernels,
// whole rows per workgroup.  Its cos/sin are the packed float32 values the
// host derives in float64, as pq_rotate's kernel derives them on the device,
// and its layer arithmetic is the same, so the results equal pq_rotate's /
// pq_rotate_mxfp4's for the pairs and angles the operands were packed from.
extern "C" int pq_rotate_rows(const void* x, int x_dtype, const uint32_t* rot_idx, const float* rot_cs,
                              const float* scales, void* out, uint8_t* mx_scales, int64_t rows, int64_t h, int krot,
                              int out_mode, void* stream) {
  PQ_REQUIRE(rows >= 0 && rows <= 0x7fffffffLL && h > 0 && h % 128 == 0 && h <= 16384, PQ_ERR_ARG,
             "pq_rotate_rows: need h %% 128 == 0 and 0 < h <= 16384 (h=%lld, rows=%lld)", (long long)h,
             (long long)rows);
  PQ_REQUIRE(krot >= 1 && krot <= 16, PQ_ERR_UNSUPPORTED, "pq_rotate_rows: krot=%d not in 1..16", krot);
  PQ_REQUIRE(x_dtype == PQ_F32 || x_dtype == PQ_F16 || x_dtype == PQ_BF16, PQ_ERR_UNSUPPORTED,
             "pq_rotate_rows: x dtype code %d", x_dtype);
  PQ_REQUIRE(out_mode == PQ_ROWS_SAME || out_mode == PQ_ROWS_MXFP4, PQ_ERR_ARG, "pq_rotate_rows: out_mode %d",
             out_mode);
  if (rows == 0) return PQ_OK;
  PQ_REQUIRE(x && rot_idx && rot_cs && out && (out_mode != PQ_ROWS_MXFP4 || mx_scales), PQ_ERR_ARG,
             "pq_rotate_rows: null pointer");
  PQ_REQUIRE(pq::aligned_to(x, 16) && pq::aligned_to(rot_idx, 16) && pq::aligned_to(rot_cs, 16) &&
                 pq::aligned_to(out, 16),
             PQ_ERR_ARG, "pq_rotate_rows: x, rot_idx, rot_cs and out must be 16-byte aligned");
  pq::RotGroup grp{};
  grp.count = 1;
  grp.mem[0] = {rot_idx, rot_cs, scales, out, nullptr, mx_scales};
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int hh = static_cast<int>(h);
  switch (x_dtype) {
    case PQ_F32: pq::launch_plain_rows_f32(x, grp, rows, hh, krot, out_mode, s); break;
    case PQ_F16: pq::launch_plain_rows_f16(x, grp, rows, hh, krot, out_mode, s); break;
    default: pq::launch_plain_rows_bf16(x, grp, rows, hh, krot, out_mode, s); break;
  }
  return pq::launch_status("pq_rotate_rows launch");
}

extern "C" int pq_rotate_quant_i8(const void* x, int x_dtype, const uint32_t* rot_idx, const float* rot_cs,
                                  const float* scales, int8_t* xq, float* xscale, void* xrot, int64_t rows,
                                  int64_t h, int krot, unsigned flags, void* stream) {
  PQ_REQUIRE(rows >= 0 && rows <= 0x7fffffffLL && h > 0 && h % 128 == 0 && h <= 16384, PQ_ERR_ARG,
             "pq_rotate_quant_i8: need h %% 128 == 0 and 0 < h <= 16384 (h=%lld, rows=%lld)", (long long)h,
             (long long)rows);
  PQ_REQUIRE(krot >= 1 && krot <= 16, PQ_ERR_UNSUPPORTED, "pq_rotate_quant_i8: krot=%d not in 1..16", krot);
  PQ_REQUIRE(x_dtype == PQ_F32 || x_dtype == PQ_F16 || x_dtype == PQ_BF16, PQ_ERR_UNSUPPORTED,
             "pq_rotate_quant_i8: dtype code %d", x_dtype);
  PQ_REQUIRE((flags & ~(PQ_RQ_INPUT_FP16 | PQ_RQ_MATERIALIZE_FP16)) == 0, PQ_ERR_ARG,
             "pq_rotate_quant_i8: unknown flags 0x%x", flags);
  if (rows == 0) return PQ_OK;
  PQ_REQUIRE(x && rot_idx && rot_cs && xq && xscale, PQ_ERR_ARG, "pq_rotate_quant_i8: null pointer");
  PQ_REQUIRE(pq::aligned_to(x, 16) && pq::aligned_to(xq, 8) && pq::aligned_to(rot_idx, 16) &&
                 pq::aligned_to(rot_cs, 16) && (xrot == nullptr || pq::aligned_to(xrot, 16)),
             PQ_ERR_ARG,
             "pq_rotate_quant_i8: x, rot_idx, rot_cs and xrot must be 16-byte aligned, xq 8-byte aligned");
  pq::RotGroup grp{};
  grp.count = 1;
  grp.mem[0] = {rot_idx, rot_cs, scales, xq, xscale, xrot};
  pq::launch_rotate_quant_group(x, x_dtype, grp, rows, static_cast<int>(h), krot, flags,
                                static_cast<hipStream_t>(stream));
  return pq::launch_status("pq_rotate_quant_i8 launch");
}

extern "C" int pq_quant_i8(const void* x, int x_dtype, int8_t* xq, float* xscale, int64_t rows, int64_t h,
                           void* stream) {
  PQ_REQUIRE(rows >= 0 && h > 0 && h % 8 == 0 && h <= (1 << 24), PQ_ERR_ARG,
             "pq_quant_i8: need h %% 8 == 0 (h=%lld)", (long long)h);
  PQ_REQUIRE(x_dtype == PQ_F32 || x_dtype == PQ_F16 || x_dtype == PQ_BF16, PQ_ERR_UNSUPPORTED,
             "pq_quant_i8: dtype code %d", x_dtype);
  if (rows == 0) return PQ_OK;
  PQ_REQUIRE(x && xq && xscale, PQ_ERR_ARG, "pq_quant_i8: null pointer");
  PQ_REQUIRE(pq::aligned_to(x, 16) && pq::aligned_to(xq, 8), PQ_ERR_ARG,
             "pq_quant_i8: x must be 16-byte and xq 8-byte aligned");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int hh = static_cast<int>(h);
  switch (x_dtype) {
    case PQ_F32: launch_quant<PQ_F32>(x, xq, xscale, rows, hh, s); break;
    case PQ_F16: launch_quant<PQ_F16>(x, xq, xscale, rows, hh, s); break;
    default: launch_quant<PQ_BF16>(x, xq, xscale, rows, hh, s); break;
  }
  return pq::launch_status("pq_quant_i8 launch");
}
