// The dense linear's product for more rows: (bitrate, codebook) (2, 2), (3, 2).
#include "linear_rows.cuh"

namespace exl3 {
template void linear_rows_product<2, 2>(const LinearRowsArgs& a, int width, float* part, void* out, int out_dt,
                                         int64_t out_stride, hipStream_t s);
template void linear_rows_product<3, 2>(const LinearRowsArgs& a, int width, float* part, void* out, int out_dt,
                                         int64_t out_stride, hipStream_t s);
}  // namespace exl3
