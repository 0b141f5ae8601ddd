// Launchers shared between the library's translation units (not exported).
#ifndef PQ_INTERNAL_H
#define PQ_INTERNAL_H

#include "pq_common.h"

#define PQ_HIDDEN __attribute__((visibility("hidden")))

namespace pq {

// Linears that share one input run as a group: one rotation launch and one
// GEMM launch over the members' concatenated output columns.
constexpr int kMaxGroup = 4;

// One member of a GEMM group: its A operand (int8 rows xq + token scales xs,
// or rotated rows xr + per-group maxima gmax), its packed weights, its bias
// and its output y [m][n].  The partials instances of the kernels (the
// parity entry points) write, instead of y, the member's int32 partials
// [m][k/128][n] and, when the kernel quantizes A itself, the int8 image of A
// it multiplies (a_out [m][k]) and the token scales of its epilogue
// (as_out [m]).
struct GemmMember {
  const int8_t* xq;
  const float* xs;
  const void* xr;
  const float* gmax;
  const uint8_t* wpack;
  const uint32_t* wmeta;
  const void* bias;
  void* y;
  int n;
  int32_t* partials;
  int8_t* a_out;
  float* as_out;
};
struct GemmGroup {
  GemmMember mem[kMaxGroup];
  int count;
  int first[kMaxGroup + 1];   // first workgroup tile of each member; set by the launchers
};

// One member of a rotation group (grid.y = member): its rotation operands,
// its outputs -- out / out_scale = xr / gmax for the split rotation, xq /
// xscale for the row rotate+quant -- and an optional fp16 copy of the
// rotated rows (xrot, row kernel only).
struct RotMember {
  const uint32_t* rot_idx;
  const float* rot_cs;
  const float* scales;
  void* out;
  float* out_scale;
  void* xrot;
  int tiled;   // row kernel: rows m of the tiled order (pqd::a_tile_offset, a16_tile_offset) of the int8 codes
               // and of the fp16 rows; 0: row-major
};
struct RotGroup {
  RotMember mem[kMaxGroup];
  int count;
};

// Per-token int8 quantization of a split rotation's output (launch_quant_split):
// xr [m][k] (fp16 or fp32) and gmax [m][k/128] in, xq [m][k] and xscale [m] out.
struct QuantMember {
  const void* xr;
  const float* gmax;
  int8_t* xq;
  float* xscale;
};
struct QuantGroup {
  QuantMember mem[kMaxGroup];
  int count;
  int tiled;   // rows m of the tiled order (pqd::a_tile_offset) for xq; 0: row-major
};

// Rows per launch of the split rotation (and rows the rotated GEMM accepts).
constexpr int kSplitMaxRows = 16;

// Optional RMSNorm prologue of a group's rotation (a decoder layer's norm in
// front of q/k/v or gate/up):  s = x + res (rounded to x's dtype; s = x when
// res is null),  h = round(w * round(s * rsqrt(mean_k(s^2) + eps))), both
// roundings to x's dtype, mean and rsqrt in float32.  The members rotate h;
// h and s are also written when h_out / s_out are set ([m][k], x's dtype).
// w: [k] in x's dtype.
//
// mode generalizes the prologue (PQ_PRO_*): RMSNORM as above; ADD rotates
// s = x + res (rounded to x's dtype) and writes it to s_out when set; SWIGLU
// rotates h = round(round(silu(x)) * res) (silu in float32: x / (1 + exp(-x)))
// and writes it to h_out when set.
struct NormArgs {
  const void* res;
  const void* w;
  void* h_out;
  void* s_out;
  float eps;
  int mode;
};

// The prologue arguments of the fused group entry points, checked.
PQ_HIDDEN int prologue_args(const char* who, const void* x2, const void* norm_weight, float eps, int mode,
                            void* h_out, void* sum_out, int x_dtype, int64_t m, NormArgs* out);

// Rotation of m <= kSplitMaxRows rows with one wave per 128-channel group,
// for every member of the group: xr [m][h] rotated values (fp16 when flags
// has PQ_RQ_MATERIALIZE_FP16, else fp32) and gmax [m][h/128] the absmax of
// each row's group.
// rows_per_wave > 0 spreads the m rows over ceil(m / rows_per_wave) waves
// per group (each wave then holds at most rows_per_wave rows); 0 keeps all
// m <= kSplitMaxRows rows in one wave.
PQ_HIDDEN void launch_rotate_split(const void* x, int x_dtype, const RotGroup& grp, int m, int h, int krot,
                                   unsigned flags, hipStream_t stream, const NormArgs* norm = nullptr,
                                   int rows_per_wave = 0);
// Token scales (absmax / 127 over each row's group maxima) and int8 codes of
// a split rotation's rows; the same values the rotated decode GEMM derives in
// its prologue.  mat16: xr holds fp16 (else fp32).
PQ_HIDDEN void launch_quant_split(const QuantGroup& grp, int m, int h, bool mat16, hipStream_t stream);
// Rotation + per-token int8 quant of whole rows for every member of the group.
PQ_HIDDEN void launch_rotate_quant_group(const void* x, int x_dtype, const RotGroup& grp, int64_t rows, int h,
                                         int krot, unsigned flags, hipStream_t stream,
                                         const NormArgs* norm = nullptr);

// launch_rotate_quant_group and the plain / MXFP4 rows of pq_rotate_rows
// (grp.count = 1) for one input dtype (pq_rows.h).
#define PQ_ROWS_DECL(dt)                                                                                              \
  PQ_HIDDEN void launch_rows_##dt(const void* x, const RotGroup& grp, int64_t rows, int h, int krot, unsigned flags,  \
                                  hipStream_t stream, const NormArgs* norm);                                          \
  PQ_HIDDEN void launch_plain_rows_##dt(const void* x, const RotGroup& grp, int64_t rows, int h, int krot,            \
                                        int out_mode, hipStream_t stream);
PQ_ROWS_DECL(f32)
PQ_ROWS_DECL(f16)
PQ_ROWS_DECL(bf16)
#undef PQ_ROWS_DECL

// Decode GEMM whose A operand is quantized in the kernel from launch_rotate_split's
// output: token scale = max over the row's gmax / 127.  Returns false when m or
// the LDS image of A (m x (k + 16) bytes) is out of range.
PQ_HIDDEN bool gemm_rotated_supported(int64_t m, int64_t k);
// The GEMM of a group (count >= 1 members, same m and k).  aq selects the A
// operand: 0 = xq/xs (any m), 1 / 2 = fp16 / fp32 xr plus gmax quantized in
// the kernel (gemm_rotated_supported(m, k)).
PQ_HIDDEN void launch_gemm_group(GemmGroup grp, int aq, int bias_dtype, int y_dtype, int m, int k,
                                 hipStream_t stream);
// launch_gemm_group's kernels, with the same configuration and tiling, in
// their partials form: each member's int32 partials (and, for aq != 0, its
// A image and token scales) go to the member's partials / a_out / as_out.
PQ_HIDDEN void launch_gemm_group_partials(GemmGroup grp, int aq, int m, int k, hipStream_t stream);

// The GEMM behind the quantizers of a group of m rows: kNone that of launch_gemm_group, kTiled the mid-size GEMM on
// tiled int8 codes (xq in the order of pqd::a_tile_offset), kChains the prefill tiles on row-major codes, summing in
// the mid-size GEMM's order.
//
// From kMidFixedRows + 1 rows on, a row's outputs must not depend on which linears share its launch (a group
// returns the bits its members return when called one by one), so there the order of the sum over K is fixed by m
// and k (gemm_mid_waves: the waves of the mid-size GEMM that split K, or 0: the one chain of launch_gemm_group).
// The prefill tiles can take the place of the mid-size GEMM's kMidChains waves, not of eight, which are for few rows.
//
// Up to 96 rows eight waves leave fewer CUs idle (on fewer than 16 groups of K their final sum costs more than that).
// Past 256 rows a wide launch is best on 192 x 256 tiles, which have no room for chains (gate and up, N = 24576, K =
// 4096, M = 320: 72 us in one chain, 81 to 103 in four), so only short rows (small hidden sizes: few columns too; to
// 384 rows) and long ones (down: N = 4096, K = 12288, M = 320: 71 us on the prefill tiles, 51 here) stay.
// Two decoder layers in us, all sizes in one chain / by this rule / four chains for every K: hidden 1536 / MLP 3840
// M = 300 175 / 160 / 148, 4096 / 12288 M = 300 474 / 426 / 469.
constexpr int kMidFixedRows = 64, kMidMaxRows = 512, kMidChains = 4;
constexpr int gemm_mid_waves(int64_t m, int64_t k) {
  if (k < 1024 || m > (k >= 6144 ? kMidMaxRows : k <= 3072 ? 384 : 256)) return 0;
  return m <= 96 && k >= 2048 ? 8 : kMidChains;
}
enum class MidGemm { kNone, kTiled, kChains };
PQ_HIDDEN MidGemm gemm_mid_choice(const GemmGroup& grp, int64_t m, int64_t k);
// Time (us) of launch_gemm_chains less the fixed part of the mid-size GEMM's, fitted to launches of 65 to 512 rows
// at K = 1024 to 12288.
PQ_HIDDEN double gemm_chains_us(const GemmGroup& grp, int64_t m, int64_t k);
PQ_HIDDEN void launch_gemm_chains(const GemmGroup& grp, int bias_dtype, int y_dtype, int m, int k, hipStream_t stream);
PQ_HIDDEN void launch_gemm_chains_partials(const GemmGroup& grp, int m, int k, hipStream_t stream);
PQ_HIDDEN void launch_gemm_mid(const GemmGroup& grp, int bias_dtype, int y_dtype, int m, int k, hipStream_t stream);
PQ_HIDDEN void launch_gemm_mid_partials(const GemmGroup& grp, int m, int k, hipStream_t stream);
// Row-major copy [m][k] of tiled codes.
PQ_HIDDEN void launch_untile_a(const int8_t* tiled, int8_t* out, int m, int k, hipStream_t stream);

}  // namespace pq

#endif
