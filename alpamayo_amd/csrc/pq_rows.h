// Rotation + per-token int8 quantization of whole rows per workgroup (and the
// same rotation with plain or MXFP4 output): kernel and launch templates.
// Instantiated for one input dtype each by pq_rows_f32.hip, pq_rows_f16.hip
// and pq_rows_bf16.hip, which compile in parallel.  Semantics and float32
// operation order: pq_rotate.hip.
#pragma once

#include <algorithm>
#include <type_traits>

#include "pq_device.h"
#include "pq_internal.h"

using pqd::quant4;

namespace {

// ---------------------------------------------------------------------------
// Fused rotate + quant over blocks of RB rows (RB a compile-time constant, so
// the RB rows are RB independent register chains with no per-row branches).
// 512 threads; wave w rotates groups w, w+8, ... for the block's rows: lane l
// loads channels l and l+64 of each row (coalesced) and runs the packed
// register chain (one cross-lane fetch per layer, no LDS traffic inside the
// layers), then stores the finished values into a row buffer [RB][h] (fp16
// when the result is materialized in fp16, fp32 otherwise).  The next group's
// parameters and inputs are requested before the current group's layers run.
// After a block-wide absmax per row the row buffer is quantized with
// coalesced stores.  Parameters are read once per group per RB rows.
// ---------------------------------------------------------------------------
constexpr int kRQWaves = 8;

//
// With NORM the rows first go through the prologue of nm.mode (PQ_PRO_*):
// RMSNORM computes the RMSNorm factor of each of the block's rows (wave r
// takes row r, with the same per-row routine as the split rotation) and
// rotates the normalized values; ADD rotates x + res; SWIGLU rotates
// silu(x) * up.  Member 0's blocks also write h / the residual sum s when
// asked.
//
// OUT selects what the block writes: kRqInt8 the int8 codes and token
// scales (and the fp16 rows when asked); kRqRows the rotated rows in x's
// dtype (the rotation::rotate result); kRqMxfp4 their OCP MXFP4 codes and
// E8M0 scales (mb.out / mb.xrot, the rotation::rotate_and_quant_mxfp4
// result).  The last two take no prologue, no fp16 rounding and no flags.
//
// IN fixes how the input reaches the rotation: kInAsIs as it is, kInF16
// rounded to fp16 (PQ_RQ_INPUT_FP16; the rounding and the channel scale
// then cost one v_cvt_f16_f32 and one v_fma_mix_f32), kInFlag as the flag
// says at run time.
//
// With MAT16 the row buffer is channel-major: channel c's RB fp16 values lie
// side by side at rowbuf[c * RB], so a lane stores a slot's RB rows with
// RB / 2 packed converts and one LDS write.
constexpr int kRqInt8 = 0, kRqRows = 1, kRqMxfp4 = 2;
constexpr int kInAsIs = 0, kInF16 = 1, kInFlag = 2;

template <int DT, int KP, bool MAT16, int RB, bool NORM, int OUT = kRqInt8, int IN = kInFlag>
__global__ __launch_bounds__(kRQWaves * 64) void rotate_quant_kernel(const void* __restrict__ x,
                                                                       const pq::RotGroup grp, int64_t row_begin,
                                                                       int h, int krot, unsigned flags,
                                                                       const pq::NormArgs nm) {
  static_assert(RB <= kRQWaves, "one wave per row for the norm factors");
  static_assert(OUT == kRqInt8 || (!MAT16 && !NORM), "plain and MXFP4 outputs come from the float32 rows");
  const pq::RotMember& mb = grp.mem[blockIdx.y];
  const uint32_t* __restrict__ rot_idx = mb.rot_idx;
  const float* __restrict__ rot_cs = mb.rot_cs;
  const float* __restrict__ scales = mb.scales;
  int8_t* __restrict__ xq = static_cast<int8_t*>(mb.out);
  float* __restrict__ xscale = mb.out_scale;
  uint16_t* __restrict__ xrot = static_cast<uint16_t*>(mb.xrot);
  const int tiled = mb.tiled;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  __shared__ float red[kRQWaves][RB];
  using RowT = typename std::conditional<MAT16, uint16_t, float>::type;
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);   // wave-uniform: scalar branches
  const bool in16 = (flags & PQ_RQ_INPUT_FP16) != 0;
  const float nz = pqd::opaque_neg_zero();
  const int G = h >> 7;
  RowT* rowbuf = reinterpret_cast<RowT*>(lds_raw);
  const int64_t row0 = row_begin + static_cast<int64_t>(blockIdx.x) * RB;
  // Channel-scale loads stay unconditional: without scales they read
  // rot_cs[0] and the value is replaced by 1.
  const bool has_scales = scales != nullptr;
  const float* sp = has_scales ? scales : rot_cs;
  const int smask = has_scales ? 0x7fffffff : 0;

  float rmax[RB];
#pragma unroll
  for (int r = 0; r < RB; ++r) rmax[r] = 0.0f;

  // Two register sets, used alternately (the group loop is unrolled twice): the set of group g is
  // computed while the loads of group g + kRQWaves land in the other one, with no copies between them.
  pqd::RotLane<KP> rl[2];
  uint32_t xa[2][RB], xb[2][RB];
  float sa[2] = {1.0f, 1.0f}, sb[2] = {1.0f, 1.0f};
  // bfloat16 rows of the int8 path (16-byte aligned, h a multiple of 128)
  // are read as dwords: lanes 2i and 2i+1 load the same pair of channels and
  // each moves its own half into the high half of a float with one byte
  // permute (a 16-bit load costs a zero-extension here on top of the shift).
  constexpr bool kPairLoads = DT == PQ_BF16 && OUT == kRqInt8;
  const uint32_t psel = (lane & 1) ? 0x03020c0cu : 0x01000c0cu;
  static_assert(!kPairLoads || IN != kInFlag, "bfloat16 input fixes its treatment at compile time");
  auto raw_f32 = [&](uint32_t raw) -> float {
    if constexpr (kPairLoads) return __uint_as_float(__builtin_amdgcn_perm(0u, raw, psel));
    else return pq_raw_to_f32<DT>(raw);
  };
  const int lane_ch = kPairLoads ? (lane & ~1) : lane;
  // channel lane (+ c0) of the row that starts at element e0 (a multiple of 128)
  auto load_row = [&](const void* base, int64_t e0) -> uint32_t {
    if constexpr (kPairLoads) return *reinterpret_cast<const uint32_t*>(static_cast<const uint16_t*>(base) + e0 + lane_ch);
    else return pq_load_raw<DT>(base, e0 + lane_ch);
  };
  auto load_inputs = [&](int g, uint32_t (&va)[RB], uint32_t (&vb)[RB], float& s0, float& s1) {
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      va[r] = load_row(x, (row0 + r) * h + g * 128);
      vb[r] = load_row(x, (row0 + r) * h + g * 128 + 64);
    }
    s0 = sp[(g * 128 + lane) & smask];
    s1 = sp[(g * 128 + 64 + lane) & smask];
  };

  // Prologue: residual / up rows and norm weights ride along with the
  // inputs (unconditional loads; without a residual or weight they re-read x
  // and are unused).
  __shared__ float s_rinv[RB];
  const bool pro_norm = NORM && nm.mode == PQ_PRO_RMSNORM;
  const bool pro_glu = NORM && nm.mode == PQ_PRO_SWIGLU;
  const void* nres = NORM && nm.res != nullptr ? nm.res : x;
  const void* nwp = pro_norm ? nm.w : x;
  uint32_t ra[2][RB], rb[2][RB];
  uint32_t wa[2] = {0, 0}, wb[2] = {0, 0};
  auto load_norm = [&](int g, uint32_t (&va)[RB], uint32_t (&vb)[RB], uint32_t& w0, uint32_t& w1) {
    if constexpr (NORM) {
#pragma unroll
      for (int r = 0; r < RB; ++r) {
        va[r] = load_row(nres, (row0 + r) * h + g * 128);
        vb[r] = load_row(nres, (row0 + r) * h + g * 128 + 64);
      }
      w0 = pq_load_raw<DT>(nwp, g * 128 + lane);
      w1 = pq_load_raw<DT>(nwp, g * 128 + 64 + lane);
    }
  };
  // the first group's loads go out before the RMSNorm factor is reduced, so
  // they are in flight while waves 0..RB-1 sum their rows
  if (w < G) {
    pqd::load_rot_lane<KP, false>(rot_idx, rot_cs, w, lane, rl[0]);
    load_inputs(w, xa[0], xb[0], sa[0], sb[0]);
    load_norm(w, ra[0], rb[0], wa[0], wb[0]);
  }
  if (pro_norm) {
    if (w < RB) {
      const float r = pqd::rms_inv(pqd::row_sumsq<DT>(x, nm.res, (row0 + w) * h, h, lane), h, nm.eps);
      if (lane == 0) s_rinv[w] = r;
    }
    pqd::lds_barrier();   // s_rinv is written (LDS only: the loads above stay in flight)
  }
  const bool write_norm = NORM && blockIdx.y == 0;   // the same for every member: member 0 writes

  for (int g0 = w; g0 < G; g0 += 2 * kRQWaves) {
#pragma unroll
    for (int ph = 0; ph < 2; ++ph) {
      const int g = g0 + ph * kRQWaves;
      if (g >= G) break;   // wave-uniform
      const int nx = ph ^ 1;
      const int gn = (g + kRQWaves < G) ? g + kRQWaves : g;   // clamped: the loads stay unconditional
      pqd::load_rot_lane<KP, false>(rot_idx, rot_cs, gn, lane, rl[nx]);
      load_inputs(gn, xa[nx], xb[nx], sa[nx], sb[nx]);
      load_norm(gn, ra[nx], rb[nx], wa[nx], wb[nx]);

      const pqd::RotLane<KP>& cur = rl[ph];
      const bool sw = pqd::rot_init_swapped(cur);
      const float s0 = has_scales ? sa[ph] : 1.0f, s1 = has_scales ? sb[ph] : 1.0f;
      float a[RB], b[RB];
      if constexpr (kPairLoads && !NORM) {
        // The initial slot swap rides in the byte permute that unpacks the
        // bfloat16 values: with the dword of channel lane + 64 as its upper
        // source, adding 4 to the selector's two data bytes takes that
        // channel instead (two selectors per group, no select per row).
        const uint32_t to_b = sw ? 0x04040000u : 0u;
        const uint32_t sel_a = psel + to_b, sel_b = psel + (0x04040000u - to_b);
        const float sc_a = sw ? s1 : s0, sc_b = sw ? s0 : s1;
#pragma unroll
        for (int r = 0; r < RB; ++r) {
          const float va = __uint_as_float(__builtin_amdgcn_perm(xb[ph][r], xa[ph][r], sel_a));
          const float vb = __uint_as_float(__builtin_amdgcn_perm(xb[ph][r], xa[ph][r], sel_b));
          if constexpr (IN == kInF16) {
            a[r] = pqd::f16_scaled(va, sc_a, nz);
            b[r] = pqd::f16_scaled(vb, sc_b, nz);
          } else {
            a[r] = va * sc_a;
            b[r] = vb * sc_b;
          }
        }
      } else {
#pragma unroll
        for (int r = 0; r < RB; ++r) {
          float lo = raw_f32(xa[ph][r]), hi = raw_f32(xb[ph][r]);
          if constexpr (NORM) {
            const int64_t ro = (row0 + r) * h + g * 128 + lane;
            if (pro_glu) {
              lo = pqd::swiglu<DT>(lo, raw_f32(ra[ph][r]));
              hi = pqd::swiglu<DT>(hi, raw_f32(rb[ph][r]));
            } else {
              if (nm.res != nullptr) {
                lo = pqd::round_to_dt<DT>(lo + raw_f32(ra[ph][r]));
                hi = pqd::round_to_dt<DT>(hi + raw_f32(rb[ph][r]));
              }
              if (write_norm && nm.s_out != nullptr) {
                pq_store_from_f32<DT>(nm.s_out, ro, lo);
                pq_store_from_f32<DT>(nm.s_out, ro + 64, hi);
              }
              if (pro_norm) {
                lo = pqd::rms_apply<DT>(lo, s_rinv[r], pq_raw_to_f32<DT>(wa[ph]));
                hi = pqd::rms_apply<DT>(hi, s_rinv[r], pq_raw_to_f32<DT>(wb[ph]));
              }
            }
            if ((pro_norm || pro_glu) && write_norm && nm.h_out != nullptr) {
              pq_store_from_f32<DT>(nm.h_out, ro, lo);
              pq_store_from_f32<DT>(nm.h_out, ro + 64, hi);
            }
          }
          if constexpr (IN == kInF16) {
            lo = pqd::f16_scaled(lo, s0, nz);
            hi = pqd::f16_scaled(hi, s1, nz);
          } else if constexpr (IN == kInFlag) {
            lo = (in16 ? pq_round_f16(lo) : lo) * s0;
            hi = (in16 ? pq_round_f16(hi) : hi) * s1;
          } else {
            lo = lo * s0;
            hi = hi * s1;
          }
          a[r] = sw ? hi : lo;
          b[r] = sw ? lo : hi;
        }
      }
      pqd::rot_layers<KP, RB>(cur, krot, a, b);
      const int fa = g * 128 + pqd::rot_final_a(cur), fb = g * 128 + pqd::rot_final_b(cur);
      if constexpr (MAT16) {   // (24-bit multiplies: full rate for 3 and 6 rows too)
        pqd::store_f16xn<RB>(rowbuf + __umul24(fa, RB), a);
        pqd::store_f16xn<RB>(rowbuf + __umul24(fb, RB), b);
      }
#pragma unroll
      for (int r = 0; r < RB; ++r) {
        const float vi = a[r], vj = b[r];
        if constexpr (!MAT16) {
          rowbuf[r * h + fa] = vi;
          rowbuf[r * h + fb] = vj;
        }
        // the float32 values: rounding to fp16 is monotonic, so the row's
        // fp16 absmax is its float32 absmax rounded once (below)
        rmax[r] = fmaxf(rmax[r], fmaxf(fabsf(vi), fabsf(vj)));
      }
    }
  }

  if constexpr (OUT == kRqRows) {
    // the rotated rows in x's dtype, 8 elements (16 or 32 bytes) per thread per step
    __syncthreads();
    const int per_row = h >> 3;
    for (int e = t; e < RB * per_row; e += kRQWaves * 64) {
      const int r = e / per_row;
      const int c8 = (e - r * per_row) * 8;
      const float* src = reinterpret_cast<const float*>(rowbuf) + r * h + c8;
      const float4 a = *reinterpret_cast<const float4*>(src);
      const float4 b = *reinterpret_cast<const float4*>(src + 4);
      const int64_t o = (row0 + r) * h + c8;
      if constexpr (DT == PQ_F32) {
        float* dst = static_cast<float*>(mb.out) + o;
        *reinterpret_cast<float4*>(dst) = a;
        *reinterpret_cast<float4*>(dst + 4) = b;
      } else {
        const float f[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        uint32_t wd[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint32_t lo = DT == PQ_F16 ? pq_f32_to_f16(f[2 * q]) : pq_f32_to_bf16(f[2 * q]);
          const uint32_t hi = DT == PQ_F16 ? pq_f32_to_f16(f[2 * q + 1]) : pq_f32_to_bf16(f[2 * q + 1]);
          wd[q] = lo | (hi << 16);
        }
        *reinterpret_cast<uint4*>(static_cast<uint16_t*>(mb.out) + o) = make_uint4(wd[0], wd[1], wd[2], wd[3]);
      }
    }
    return;
  } else if constexpr (OUT == kRqMxfp4) {
    // 32-channel blocks: 4 consecutive threads of 8 channels each exchange their absmax
    __syncthreads();
    const int per_row = h >> 3;
    uint8_t* __restrict__ codes = static_cast<uint8_t*>(mb.out);
    uint8_t* __restrict__ mxs = static_cast<uint8_t*>(mb.xrot);
    for (int e0 = 0; e0 < RB * per_row; e0 += kRQWaves * 64) {   // uniform trip count: the shuffles see every lane
      const int e = e0 + t;
      const bool live = e < RB * per_row;
      const int ee = live ? e : 0;
      const int r = ee / per_row;
      const int c8 = (ee - r * per_row) * 8;
      const float* src = reinterpret_cast<const float*>(rowbuf) + r * h + c8;
      const float4 a = *reinterpret_cast<const float4*>(src);
      const float4 b = *reinterpret_cast<const float4*>(src + 4);
      const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
      float am = 0.0f;
      bool nan = false;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        am = fmaxf(am, fabsf(v[q]));
        nan = nan || (v[q] != v[q]);
      }
      am = fmaxf(am, __shfl_xor(am, 1));
      am = fmaxf(am, __shfl_xor(am, 2));
      int nn = nan ? 1 : 0;
      nn |= __shfl_xor(nn, 1);
      nn |= __shfl_xor(nn, 2);
      const int ex = pqd::mx_shared_exp(am);
      const float inv = pqd::mx_inv_scale(ex);
      uint32_t wd = 0;
#pragma unroll
      for (int q = 0; q < 8; ++q) wd |= pqd::mx_e2m1(v[q] * inv) << (4 * q);
      if (live) {
        const int64_t row = row0 + r;
        *reinterpret_cast<uint32_t*>(codes + row * (h >> 1) + (c8 >> 1)) = wd;
        if ((c8 & 31) == 0) mxs[row * (h >> 5) + (c8 >> 5)] = nn ? 0xFFu : static_cast<uint8_t>(ex + 127);
      }
    }
    return;
  }

  uint32_t ubits[RB];   // the rows' maxima are >= 0: their bits order like unsigned integers
#pragma unroll
  for (int r = 0; r < RB; ++r) ubits[r] = __float_as_uint(rmax[r]);
  pq_wave_umax_n<RB>(ubits);
  if (lane == 0) {
#pragma unroll
    for (int r = 0; r < RB; ++r) red[w][r] = __uint_as_float(ubits[r]);
  }
  __syncthreads();
  // Each row's 127 / absmax, and its token scale, once per row.
  __shared__ float s_inv[RB];
  if (t < RB) {
    float am = 0.0f;
#pragma unroll
    for (int ww = 0; ww < kRQWaves; ++ww) am = fmaxf(am, red[ww][t]);
    if constexpr (MAT16) am = pq_round_f16(am);   // = the absmax of the fp16 rows
    s_inv[t] = pqd::inv_scale(am);
    if (xq != nullptr) xscale[row0 + t] = am / 127.0f;   // null: only the fp16 rows are wanted (W4A16)
  }
  __syncthreads();

  if constexpr (MAT16) {
    // Quantize the channel-major fp16 buffer: a thread takes 8 channels of all
    // RB rows (RB 16-byte reads), then writes each row's 8 codes (8 bytes,
    // coalesced across the threads) and, when asked, its 8 fp16 values.
    for (int e = t; e < (h >> 3); e += kRQWaves * 64) {
      const int c8 = e * 8;
      uint32_t d[4 * RB];   // (channel c8 + k, row r) is fp16 number k * RB + r of d
      const uint4* src = reinterpret_cast<const uint4*>(rowbuf + c8 * RB);
#pragma unroll
      for (int q = 0; q < RB; ++q) {
        const uint4 u = src[q];
        d[4 * q] = u.x;
        d[4 * q + 1] = u.y;
        d[4 * q + 2] = u.z;
        d[4 * q + 3] = u.w;
      }
#pragma unroll
      for (int r = 0; r < RB; ++r) {
        const int64_t ro = (row0 + r) * h + c8;
        if (xrot != nullptr) {
          uint32_t w[4];
#pragma unroll
          for (int m = 0; m < 4; ++m) w[m] = pqd::f16_pair(d, 2 * m * RB + r, (2 * m + 1) * RB + r);
          *reinterpret_cast<uint4*>(xrot + (tiled ? pqd::a16_tile_offset(row0 + r, c8, tiled, G) : ro)) =
              make_uint4(w[0], w[1], w[2], w[3]);
        }
        if (xq != nullptr) {
          const float inv = s_inv[r];
          uint32_t c[8];
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            const int i = k * RB + r;
            c[k] = pqd::quant_scaled(pqd::mul_f16(d[i >> 1], (i & 1) != 0, inv));
          }
          *reinterpret_cast<uint2*>(xq + (tiled ? pqd::a_tile_offset(row0 + r, c8, tiled, G) : ro)) =
              make_uint2(pqd::pack4(c[0], c[1], c[2], c[3]), pqd::pack4(c[4], c[5], c[6], c[7]));
        }
      }
    }
  } else {
    // Quantize the row buffer: 8 elements per thread per step.
    const int per_row = h >> 3;
    for (int e = t; e < RB * per_row; e += kRQWaves * 64) {
      const int r = e / per_row;
      const int c8 = (e - r * per_row) * 8;
      const float inv = s_inv[r];
      float f[8];
      const float4 a = *reinterpret_cast<const float4*>(rowbuf + r * h + c8);
      const float4 b = *reinterpret_cast<const float4*>(rowbuf + r * h + c8 + 4);
      f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w;
      f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
      if (xrot != nullptr) {
        uint4 o;
        o.x = pqd::pk_f16(f[0], f[1]);
        o.y = pqd::pk_f16(f[2], f[3]);
        o.z = pqd::pk_f16(f[4], f[5]);
        o.w = pqd::pk_f16(f[6], f[7]);
        *reinterpret_cast<uint4*>(xrot + (tiled ? pqd::a16_tile_offset(row0 + r, c8, tiled, G)
                                                    : (row0 + r) * h + c8)) = o;
      }
      if (xq != nullptr) {
        uint2 o;
        o.x = quant4(f[0], f[1], f[2], f[3], inv);
        o.y = quant4(f[4], f[5], f[6], f[7], inv);
        *reinterpret_cast<uint2*>(xq + (tiled ? pqd::a_tile_offset(row0 + r, c8, tiled, G) : (row0 + r) * h + c8)) = o;
      }
    }
  }
}

// Rows per block: more rows per block read the parameters fewer times, fewer
// keep enough blocks in flight; the row buffer stays within 96 KB.  Two rows
// up to 2048 rows (K = 4096, M = 1264: 15.4 -> 13.8 us against four), four
// from there (M = 3072: 21.8 us against 24.4 us with two, 28.7 us with eight),
// eight from 4096.  The fp16-row kernel from 2048 rows chooses by how its
// blocks fill the chip (rq_rows_fp16).
inline int rq_rows_per_block(int64_t rows, int h, bool mat16) {
  int rb = rows >= 4096 ? 8 : rows >= 2048 ? 4 : rows >= 256 ? 2 : 1;
  while (rb > 1 && static_cast<int64_t>(rb) * h * (mat16 ? 2 : 4) > 96 * 1024) rb >>= 1;
  return rb;
}

template <int DT, int KP, bool MAT16, int RB, bool NORM, int OUT, int IN>
void launch_rq_rb(const void* x, const pq::RotGroup& grp, int64_t row_begin, int64_t nblocks, int h, int krot,
                  unsigned flags, const pq::NormArgs& nm, hipStream_t stream) {
  if (nblocks <= 0) return;
  const size_t lds = static_cast<size_t>(RB) * h * (MAT16 ? 2 : 4);
  const dim3 grid(static_cast<unsigned>(nblocks), static_cast<unsigned>(grp.count));
  rotate_quant_kernel<DT, KP, MAT16, RB, NORM, OUT, IN><<<grid, kRQWaves * 64, lds, stream>>>(x, grp, row_begin,
                                                                                              h, krot, flags, nm);
}

// The device's CU count and LDS bytes per CU (queried once; 0 if unknown).
struct CuInfo {
  int cus = 0;
  int lds = 0;
};
inline CuInfo cu_info() {
  static const CuInfo info = [] {
    CuInfo c;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&c.cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipDeviceGetAttribute(&c.lds, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, dev) != hipSuccess)
      c = CuInfo{};
    return c;
  }();
  return info;
}

// Blocks of one fp16-row instance that registers and waves allow per CU
// (the runtime's occupancy calculator without the row buffer), queried once.
template <int DT, int KP, int RB, bool NORM, int IN>
int rq_blocks_per_cu_regs() {
  static const int n = [] {
    int b = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, rotate_quant_kernel<DT, KP, true, RB, NORM, kRqInt8, IN>,
                                                     kRQWaves * 64, 0) != hipSuccess)
      b = 0;
    return b;
  }();
  return n;
}

// Rows per block of the fp16-row kernel from 2048 rows: every block of a
// launch is equal work, so the launch takes as many rounds as its blocks
// fill on the chip (CUs x blocks per CU), and a part-filled last round costs
// nearly a full one.  Among 8, 6, 4, 3 and 2 rows, with at least two blocks
// (16 waves) per CU and a row buffer within 96 KB, take the one whose blocks
// fill their rounds best; a smaller one only when it fills them better by
// more than 2 %, since more rows per block read the layer parameters fewer
// times.  At 3072 rows: 6 rows for K = 4096 (512 blocks, one round: 21.4 ->
// 21.2 us; the prefill layer 0.871 / 0.880 -> 0.857 / 0.860 ms), 3 for
// K = 12288 (2 rounds of 2 blocks per CU: 58.0 / 58.8 -> 51.5 / 51.6 us
// against 4 rows, whose 96 KB row buffer leaves one block per CU).
template <int DT, int KP, bool NORM, int IN>
int rq_rows_fp16(int64_t rows, int h, int members) {
  const CuInfo ci = cu_info();
  if (rows < 2048 || ci.cus <= 0 || ci.lds <= 0) return rq_rows_per_block(rows, h, true);
  const int cand[5] = {8, 6, 4, 3, 2};
  const int regs[5] = {rq_blocks_per_cu_regs<DT, KP, 8, NORM, IN>(), rq_blocks_per_cu_regs<DT, KP, 6, NORM, IN>(),
                       rq_blocks_per_cu_regs<DT, KP, 4, NORM, IN>(), rq_blocks_per_cu_regs<DT, KP, 3, NORM, IN>(),
                       rq_blocks_per_cu_regs<DT, KP, 2, NORM, IN>()};
  int best = 0;
  double best_fill = -1.0;
  for (int i = 0; i < 5; ++i) {
    const int64_t lds = static_cast<int64_t>(cand[i]) * h * 2;
    if (lds > 96 * 1024) continue;
    const int64_t per_cu = std::min<int64_t>(regs[i], ci.lds / (lds + 1024));   // + the static LDS
    if (per_cu < 2) continue;
    const int64_t blocks = rows / cand[i] * members;
    const int64_t cap = per_cu * ci.cus;
    const int64_t rounds = (blocks + cap - 1) / cap;
    const double fill = static_cast<double>(blocks) / static_cast<double>(rounds * cap);
    if (fill > best_fill + 0.02) {
      best = cand[i];
      best_fill = fill;
    }
  }
  return best > 0 ? best : rq_rows_per_block(rows, h, true);
}

template <int DT, int KP, bool MAT16, bool NORM, int OUT, int IN>
void launch_rq_in(const void* x, const pq::RotGroup& grp, int64_t rows, int h, int krot, unsigned flags,
                  const pq::NormArgs& nm, hipStream_t stream) {
  int rb = 0;
  if constexpr (MAT16) rb = rq_rows_fp16<DT, KP, NORM, IN>(rows, h, grp.count);
  else rb = rq_rows_per_block(rows, h, false);
  const int64_t full = rows / rb;
  switch (rb) {
    case 8: launch_rq_rb<DT, KP, MAT16, 8, NORM, OUT, IN>(x, grp, 0, full, h, krot, flags, nm, stream); break;
    case 4: launch_rq_rb<DT, KP, MAT16, 4, NORM, OUT, IN>(x, grp, 0, full, h, krot, flags, nm, stream); break;
    case 2: launch_rq_rb<DT, KP, MAT16, 2, NORM, OUT, IN>(x, grp, 0, full, h, krot, flags, nm, stream); break;
    case 6:
      if constexpr (MAT16) launch_rq_rb<DT, KP, MAT16, 6, NORM, OUT, IN>(x, grp, 0, full, h, krot, flags, nm, stream);
      break;
    case 3:
      if constexpr (MAT16) launch_rq_rb<DT, KP, MAT16, 3, NORM, OUT, IN>(x, grp, 0, full, h, krot, flags, nm, stream);
      break;
    default: break;
  }
  const int64_t done = rb > 1 ? full * rb : 0;   // the remaining rows, one block each
  launch_rq_rb<DT, KP, MAT16, 1, NORM, OUT, IN>(x, grp, done, rows - done, h, krot, flags, nm, stream);
}

// The input treatment as a compile-time choice: an fp16 input is already
// fp16 (its prologue rounds to x's dtype as well), a bfloat16 one gets an
// instance per flag value, float32 reads the flag at run time.  The plain and
// MXFP4 outputs take no flags.
template <int DT, int KP, bool MAT16, bool NORM, int OUT = kRqInt8>
void launch_rq(const void* x, const pq::RotGroup& grp, int64_t rows, int h, int krot, unsigned flags,
               const pq::NormArgs& nm, hipStream_t stream) {
  if constexpr (OUT != kRqInt8 || DT == PQ_F16) {
    launch_rq_in<DT, KP, MAT16, NORM, OUT, kInAsIs>(x, grp, rows, h, krot, flags, nm, stream);
  } else if constexpr (DT == PQ_BF16) {
    if (flags & PQ_RQ_INPUT_FP16) launch_rq_in<DT, KP, MAT16, NORM, OUT, kInF16>(x, grp, rows, h, krot, flags, nm, stream);
    else launch_rq_in<DT, KP, MAT16, NORM, OUT, kInAsIs>(x, grp, rows, h, krot, flags, nm, stream);
  } else {
    launch_rq_in<DT, KP, MAT16, NORM, OUT, kInFlag>(x, grp, rows, h, krot, flags, nm, stream);
  }
}

// The register-chain rotation of whole rows with a plain (OUT = kRqRows) or
// MXFP4 (kRqMxfp4) output, on packed operands.
template <int DT, int OUT>
void launch_rotate_rows_dt(const void* x, const pq::RotGroup& grp, int64_t rows, int h, int krot,
                           hipStream_t stream) {
  if (krot <= 8) launch_rq<DT, 8, false, false, OUT>(x, grp, rows, h, krot, 0u, pq::NormArgs{}, stream);
  else launch_rq<DT, 16, false, false, OUT>(x, grp, rows, h, krot, 0u, pq::NormArgs{}, stream);
}

template <int DT, bool NORM>
void launch_rotate_quant_norm(const void* x, const pq::RotGroup& grp, int64_t rows, int h, int krot,
                              unsigned flags, const pq::NormArgs& nm, hipStream_t stream) {
  const bool mat16 = (flags & PQ_RQ_MATERIALIZE_FP16) != 0;
  if (krot <= 8) {
    if (mat16) launch_rq<DT, 8, true, NORM>(x, grp, rows, h, krot, flags, nm, stream);
    else launch_rq<DT, 8, false, NORM>(x, grp, rows, h, krot, flags, nm, stream);
  } else {
    if (mat16) launch_rq<DT, 16, true, NORM>(x, grp, rows, h, krot, flags, nm, stream);
    else launch_rq<DT, 16, false, NORM>(x, grp, rows, h, krot, flags, nm, stream);
  }
}

template <int DT>
void launch_rotate_quant(const void* x, const pq::RotGroup& grp, int64_t rows, int h, int krot, unsigned flags,
                         const pq::NormArgs* norm, hipStream_t stream) {
  if (norm != nullptr) launch_rotate_quant_norm<DT, true>(x, grp, rows, h, krot, flags, *norm, stream);
  else launch_rotate_quant_norm<DT, false>(x, grp, rows, h, krot, flags, pq::NormArgs{}, stream);
}

}  // namespace
