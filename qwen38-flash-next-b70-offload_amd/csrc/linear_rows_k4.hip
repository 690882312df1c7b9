// The dense linear's product for more rows: (bitrate, codebook) (4, 2), (4, 1), (4, 0).
#include "linear_rows.cuh"

namespace exl3 {
template void linear_rows_product<4, 2>(const LinearRowsArgs& a, int width, float* part, void* out, int out_dt,
                                         int64_t out_stride, hipStream_t s);
template void linear_rows_product<4, 1>(const LinearRowsArgs& a, int width, float* part, void* out, int out_dt,
                                         int64_t out_stride, hipStream_t s);
template void linear_rows_product<4, 0>(const LinearRowsArgs& a, int width, float* part, void* out, int out_dt,
                                         int64_t out_stride, hipStream_t s);
}  // namespace exl3
