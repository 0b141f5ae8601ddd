// Shared by the W4A16 kernels: operands of a linear and of a group, and the
// dequantization of the packed weights (pq_w4a16.hip).
#pragma once

#include "pq_device.h"
#include "pq_internal.h"

typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

namespace pqw16 {

struct W16Args {
  const uint16_t* x;       // fp16 [m][k]
  const uint8_t* wpack;    // packed codes
  const uint32_t* wmeta;   // s | sz << 16 per (tile, group, column)
  const void* bias;        // [n] or null
  void* y;                 // [m][n]
  int n;
};

__device__ __forceinline__ v2h as_h2(uint32_t u) { return __builtin_bit_cast(v2h, u); }
__device__ __forceinline__ uint32_t as_u32(v2h h) { return __builtin_bit_cast(uint32_t, h); }

// fp16 pairs {s, s} and {sz, sz} of a metadata word.
__device__ __forceinline__ v2h meta_s2(uint32_t meta) { return as_h2(__builtin_amdgcn_perm(meta, meta, 0x01000100u)); }
__device__ __forceinline__ v2h meta_z2(uint32_t meta) { return as_h2(__builtin_amdgcn_perm(meta, meta, 0x03020302u)); }

// One dword of codes (k order: the low nibbles of bytes 0..3, then the high
// nibbles) -> its 8 weights fp16(q * s + sz), in k order.
__device__ __forceinline__ v8h dequant8(uint32_t w, v2h s2, v2h z2) {
  const uint32_t lo = w & 0x0f0f0f0fu;
  const uint32_t hi = (w >> 4) & 0x0f0f0f0fu;
  // selector bytes 0..3 pick bytes of the second operand, 4 picks 0x64:
  // halves 0x6400 + q = 1024 + q
  constexpr uint32_t kE = 0x64646464u;
  const v2h off = {static_cast<_Float16>(1024.0f), static_cast<_Float16>(1024.0f)};
  const v2h q01 = as_h2(__builtin_amdgcn_perm(kE, lo, 0x04010400u)) - off;
  const v2h q23 = as_h2(__builtin_amdgcn_perm(kE, lo, 0x04030402u)) - off;
  const v2h q45 = as_h2(__builtin_amdgcn_perm(kE, hi, 0x04010400u)) - off;
  const v2h q67 = as_h2(__builtin_amdgcn_perm(kE, hi, 0x04030402u)) - off;
  const uint4 r = {as_u32(__builtin_elementwise_fma(q01, s2, z2)), as_u32(__builtin_elementwise_fma(q23, s2, z2)),
                   as_u32(__builtin_elementwise_fma(q45, s2, z2)), as_u32(__builtin_elementwise_fma(q67, s2, z2))};
  return __builtin_bit_cast(v8h, r);
}

// Linears that share their input, as one GEMM launch: member i owns
// workgroups first[i] .. first[i+1]-1 (set by the launcher).
struct W16Group {
  W16Args mem[pq::kMaxGroup];
  int first[pq::kMaxGroup + 1];
  int count;
};

// Mid-size GEMM on tiled fp16 rows (pqd::a16_tile_offset): whether m rows of a linear of n columns run it, alone or in
// a group (the prefill tiles sum in another order, so the choice looks at the member alone), and its launch
// (pq_w4a16_mid.hip).
PQ_HIDDEN bool w16_mid_takes(int64_t m, int64_t n, int64_t k);
// Time (us) of the prefill tiles for m > 16 rows, less the fixed part of a launch of the mid-size GEMM.
PQ_HIDDEN double w16_prefill_us(int64_t m, int64_t n, int64_t k);
PQ_HIDDEN void launch_w16_mid(const W16Group& grp, int bias_dtype, int y_dtype, int m, int k, hipStream_t stream);

}  // namespace pqw16
