// The row kernels (pq_rows.h) for f16 input.
#include "pq_rows.h"

namespace pq {
void launch_rows_f16(const void* x, const RotGroup& grp, int64_t rows, int h, int krot, unsigned flags,
                      hipStream_t stream, const NormArgs* norm) {
  launch_rotate_quant<PQ_F16>(x, grp, rows, h, krot, flags, norm, stream);
}

void launch_plain_rows_f16(const void* x, const RotGroup& grp, int64_t rows, int h, int krot, int out_mode,
                            hipStream_t stream) {
  if (out_mode == PQ_ROWS_SAME) launch_rotate_rows_dt<PQ_F16, kRqRows>(x, grp, rows, h, krot, stream);
  else launch_rotate_rows_dt<PQ_F16, kRqMxfp4>(x, grp, rows, h, krot, stream);
}
}  // namespace pq
