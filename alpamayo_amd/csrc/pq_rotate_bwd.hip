// Backward of rotation::rotate: the gradients of y = R_{K-1} ... R_0 (s * x)
// with respect to x, the angles theta and the channel scales s.
//
// Reference: RotateTensorFunc.backward (kernels/paroquant_kernels/
// interface.py:30-93), which inverts y layer by layer with one rotation launch
// per layer and gathers the pairs in torch.  Here one kernel does all layers
// (rotate_chain_bwd, pq_chain.h):
//
//   * each wave re-runs the forward layers from x in float32 and keeps every
//     layer's pair outputs (a', b') in registers -- the values the forward
//     computed, not a reconstruction from the rounded y;
//   * then it walks the layers backwards on the incoming gradient: with
//     (g_a', g_b') the gradient at layer r's output, the angle gradient is
//     g_a' b' - g_b' a' (d(a', b')/d theta = (b', -a')), and the gradient at
//     the layer's input is the transposed rotation (c g_a' - s g_b',
//     s g_a' + c g_b');
//   * below layer 0: dx = s * g_t and ds = x * g_t (t = s * x).
//
// The angle and scale gradients are sums over all rows.  A workgroup walks
// its column of row tiles grid-stride and keeps running sums in registers,
// its waves are summed through LDS in a fixed order, and each workgroup row
// writes one partial per angle / channel; a second kernel adds the partials
// in a fixed order.  The result is deterministic (no atomics).
#include <algorithm>

#include "pq_chain.h"
#include "pq_device.h"
#include "pq_internal.h"

namespace {

constexpr int kBwdRows = 16;
// Workgroup rows of the partial sums (each handles every kBwdMaxBlocks-th tile).
constexpr int64_t kBwdMaxBlocks = 64;

int64_t bwd_blocks(int64_t rows) {
  const int64_t tiles = (rows + kBwdRows - 1) / kBwdRows;
  return tiles < kBwdMaxBlocks ? tiles : kBwdMaxBlocks;
}

// grad_theta[r][P] = sum_b part_th[b][r][P]; grad_scales[c] = sum_b part_s[b][c]
// (b in order), rounded to the parameters' dtype.  nb == 0 writes zeros.
template <int DT>
__global__ __launch_bounds__(64) void rotate_bwd_reduce_kernel(const float* __restrict__ part_th,
                                                                const float* __restrict__ part_s,
                                                                void* __restrict__ g_theta,
                                                                void* __restrict__ g_scales, int nb, int n_th,
                                                                int h) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 64 + threadIdx.x;
  const bool th = i < n_th;
  if (!th && (g_scales == nullptr || i >= static_cast<int64_t>(n_th) + h)) return;
  const float* src = th ? part_th + i : part_s + (i - n_th);
  const int64_t pitch = th ? n_th : h;
  float s = 0.0f;
  int b = 0;
  for (; b + 16 <= nb; b += 16) {   // 16 partials requested at once, added in order
    float v[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) v[q] = src[(b + q) * pitch];
#pragma unroll
    for (int q = 0; q < 16; ++q) s += v[q];
  }
  for (; b < nb; ++b) s += src[b * pitch];
  if (th) pq_store_from_f32<DT>(g_theta, i, s);
  else pq_store_from_f32<DT>(g_scales, i - n_th, s);
}

template <int DT>
void launch_bwd(const void* x, const void* gy, void* gx, void* g_theta, void* g_scales, const int16_t* idx,
                const void* theta, const void* scales, int64_t rows, int h, int krot, int group, float* ws,
                hipStream_t s) {
  // The register chain where a workgroup has rows enough to pay for deriving it (tile form -> chain, us, 8 layers:
  // 128 x 4096 11.5 -> 13.0, 256 x 4096 15.8 -> 13.2, 64 x 12288 12.2 -> 11.0, 1024 x 4096 50.7 -> 22.5, 8192 x 4096
  // float32 221 -> 106; 16 layers 256 x 4096 17.6 -> 26.7, 512 x 4096 37.8 -> 31.5), a step of 32 of them at least (8
  // layers 16 x 49152 12.2 -> 17.3, 1 x 1048576 95 -> 222, 34 x 65536 25.2 -> 22.9; 16 layers 34 x 65536 47 -> 51, 49 x
  // 65536 63 -> 54), on at most one workgroup per CU (what its registers allow); else the tile form on every workgroup
  // row the workspace has room for.
  const bool chain = krot <= 8 ? rows >= 32 && rows * h >= 3 << 18 : rows >= 48 && rows * h >= 1 << 21;
  const int64_t chunks = (h + 127) / 128;
  const int nb = static_cast<int>(
      chain ? std::min<int64_t>(bwd_blocks(rows), std::max<int64_t>(1, 256 / chunks)) : bwd_blocks(rows));
  const int n_th = krot * (h / 2);
  float* part_th = ws;
  float* part_s = ws + static_cast<int64_t>(nb) * n_th;
  if (nb > 0) {
    const dim3 grid(static_cast<unsigned>(nb), static_cast<unsigned>((h + 127) / 128));
#define PQ_BWD(K_)                                                                                              \
  case K_:                                                                                                      \
    if (chain)                                                                                                  \
      pqchain::rotate_chain_bwd<DT, K_, pqchain::kWaves, true><<<grid, pqchain::kWaves * 64, 0, s>>>(           \
          x, gy, gx, idx, theta, scales, part_th, part_s, rows, h, group, krot);                                \
    else                                                                                                        \
      pqchain::rotate_chain_bwd<DT, K_, pqchain::kTileWaves, false><<<grid, pqchain::kTileWaves * 64, 0, s>>>(  \
          x, gy, gx, idx, theta, scales, part_th, part_s, rows, h, group, krot);                                \
    break;
    switch (krot) { PQ_BWD(1) PQ_BWD(2) PQ_BWD(4) PQ_BWD(8) PQ_BWD(16) }
#undef PQ_BWD
  }
  const int64_t n_out = n_th + (scales ? h : 0);
  rotate_bwd_reduce_kernel<DT><<<static_cast<unsigned>((n_out + 63) / 64), 64, 0, s>>>(
      part_th, part_s, g_theta, scales ? g_scales : nullptr, nb, n_th, h);
}

}  // namespace

extern "C" size_t pq_rotate_backward_workspace_size(int64_t rows, int64_t h, int krot) {
  if (rows < 0 || h <= 0 || krot < 1 || krot > 16) return 0;
  return static_cast<size_t>(bwd_blocks(rows)) * (static_cast<size_t>(krot) * (h / 2) + h) * sizeof(float);
}

extern "C" int pq_rotate_backward(const void* x, const void* grad_y, void* grad_x, void* grad_theta,
                                  void* grad_scales, const int16_t* idx_ij, const void* theta, const void* scales,
                                  int64_t rows, int64_t h, int krot, int group_size, int dtype, void* workspace,
                                  size_t workspace_bytes, void* stream) {
  const char* who = "pq_rotate_backward";
  PQ_REQUIRE(rows >= 0 && h > 0, PQ_ERR_ARG, "%s: rows=%lld h=%lld", who, (long long)rows, (long long)h);
  PQ_REQUIRE(group_size == 64 || group_size == 128, PQ_ERR_UNSUPPORTED,
             "%s: Unexpected group_size: %d (supported: 64, 128)", who, group_size);
  PQ_REQUIRE(krot == 1 || krot == 2 || krot == 4 || krot == 8 || krot == 16, PQ_ERR_UNSUPPORTED,
             "%s: Unsupported KROT = %d; compiled variants: 1/2/4/8/16", who, krot);
  PQ_REQUIRE(h % group_size == 0, PQ_ERR_ARG, "%s: h must be divisible by GROUP_SIZE (h=%lld, G=%d)", who,
             (long long)h, group_size);
  // (h + 127) / 128 channel blocks go on grid.y, whose limit is 65535
  PQ_REQUIRE(h <= 65535LL * 128, PQ_ERR_ARG, "%s: h=%lld too large (at most %lld)", who, (long long)h,
             65535LL * 128);
  PQ_REQUIRE(dtype == PQ_F32 || dtype == PQ_F16 || dtype == PQ_BF16, PQ_ERR_UNSUPPORTED,
             "%s: dtype code %d (Float, Half or BFloat16)", who, dtype);
  PQ_REQUIRE((rows + kBwdRows - 1) / kBwdRows <= 0x7fffffffLL, PQ_ERR_ARG, "%s: too many rows", who);
  PQ_REQUIRE(grad_theta && idx_ij && theta, PQ_ERR_ARG, "%s: null pointer", who);
  PQ_REQUIRE((scales == nullptr) == (grad_scales == nullptr), PQ_ERR_ARG,
             "%s: grad_scales must be given exactly when scales is", who);
  PQ_REQUIRE(rows == 0 || (x && grad_y && grad_x), PQ_ERR_ARG, "%s: null x / grad_y / grad_x", who);
  const size_t need = pq_rotate_backward_workspace_size(rows, h, krot);
  PQ_REQUIRE(need == 0 || (workspace != nullptr && workspace_bytes >= need && pq::aligned_to(workspace, 16)),
             PQ_ERR_WORKSPACE, "%s: a 16-byte aligned workspace of %zu bytes is needed for rows=%lld h=%lld, got %zu",
             who, need, (long long)rows, (long long)h, workspace ? workspace_bytes : (size_t)0);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int hh = static_cast<int>(h);
  float* ws = static_cast<float*>(workspace);
  switch (dtype) {
    case PQ_F32:
      launch_bwd<PQ_F32>(x, grad_y, grad_x, grad_theta, grad_scales, idx_ij, theta, scales, rows, hh, krot,
                         group_size, ws, s);
      break;
    case PQ_F16:
      launch_bwd<PQ_F16>(x, grad_y, grad_x, grad_theta, grad_scales, idx_ij, theta, scales, rows, hh, krot,
                         group_size, ws, s);
      break;
    default:
      launch_bwd<PQ_BF16>(x, grad_y, grad_x, grad_theta, grad_scales, idx_ij, theta, scales, rows, hh, krot,
                          group_size, ws, s);
      break;
  }
  return pq::launch_status("pq_rotate_backward launch");
}
