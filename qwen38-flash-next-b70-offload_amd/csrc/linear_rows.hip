// The dense EXL3 linear for more rows than the fused small path takes: out[M, n] = svh * H(sum_k xh[shard of n][m][k]
// W[k][n]) / sqrt 128 with the trellis decoded into MFMA B registers (exl3_regb.cuh), so the weights are never written
// to memory (reference: experimental/n111-victim-ring/csrc/exl3_ops.sycl:651-757; HadInKernel / HadOutKernel,
// exl3_esimd.h:286-343).
//
//   xh    input Hadamards of every (shard, row), fp16
//   rows  one workgroup per (256 or 128 columns, 16 NB rows, K-slice); with one K-slice it applies the output Hadamard
//         itself, else it stores fp32 partial sums [P][M][n] for lin_had_out_kernel
//
// Before, a call reconstructed fp16 weight slices (written and read back), multiplied them with a library GEMM into fp16
// and ran the output Hadamard over that product. 2048 -> 12,288 (4 shards), K 4, 40 rows: 111 us then (four
// reconstructions and four GEMMs of 10 us each), 26 us now, most of it the waves' serial chains and three launches
// (13.8 MB of trellis are 2.2 us at 6.3 TB/s); K 3, 1,024 rows: 160 -> 91 us (51.5 GFLOP are 21 us at the matrix cores'
// peak; the weights are decoded once per 128 rows, 19 us of VALU work); K 3, 8,192 rows: 689 -> 557 us.
#include "exl3_common.cuh"
#include "exl3_kernels.h"
#include "exl3_regb.cuh"
#include "exl3_xh.cuh"

#include <algorithm>

namespace exl3 {

// ---- input Hadamards: one wave per (4 rows, 128-block), every shard in turn (16 lanes hold a row's block, 8 values each;
// 1,024 rows of 4 shards of 2048 take 11 us, 12 us as MFMA products with H128) -----------------------------------
constexpr int kLxWaves = 8;

template <int DT>
__device__ __forceinline__ void lx_task(const LinearArgs& A, int rq, int kb) {
    const int l = lane_id(), m = rq * 4 + (l >> 4), c = kb * 128 + (l & 15) * 8;
    XRaw<DT> x;
    ld_x8<DT>(A.x, (size_t)min(m, A.M - 1) * A.x_stride + c, x);
    const float rs = row_sign() * kRsqrt128;
    for (int g = 0; g < A.S; ++g) {
        const half8_u su = ld_half8(A.suh + (size_t)g * A.k + c);
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = x_su<DT>(x, j, su[j]);
        row_fwht128_signed(v);
        half8_t o;
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = to_half(v[j] * rs);
        if (m < A.M) *(half8_t*)(A.xh + ((size_t)g * A.M + m) * A.k + c) = o;
    }
}

__global__ void __launch_bounds__(64 * kLxWaves) lin_xh_kernel(LinearArgs A) {
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kbn = A.k / 128, t = blockIdx.x * kLxWaves + wv;
    if (t >= (A.M + 3) / 4 * kbn) return;        // (whole waves: the transforms need every lane)
    if (A.x_dt == 1) lx_task<1>(A, t / kbn, t % kbn);
    else if (A.x_dt == 2) lx_task<2>(A, t / kbn, t % kbn);
    else lx_task<0>(A, t / kbn, t % kbn);
}

// ---- host --------------------------------------------------------------------------------------------------------------

// (M > 0, n a positive multiple of width)
int linear_rows_slices(int M, int k, int n, int width) {
    const int64_t rt = 16 * linear_rows_blocks(M), wgs = n / width * ((M + rt - 1) / rt);
    const int nkb = k / 128;
    // about one workgroup of 8 waves per CU: more slices cost their partial sums' traffic (40 rows, 2048 -> 12,288, K 4,
    // 48 workgroups: 1 / 2 / 4 / 8 slices 37 / 29 / 26 / 34 us; 1,024 rows, 4096 -> 2048, 64 workgroups: 84 / 58 / 48 /
    // 61 us), and up to 512 input rows a second launch for the sums costs more than the slices give (1,024 rows, 512 ->
    // 2048: 25 against 31 us)
    return nkb <= 4 ? 1 : (int)std::max<int64_t>(1, std::min<int64_t>(std::min(8, nkb / 2), 256 / wgs));
}

hipError_t launch_linear_rows(int K, int cb, const LinearRowsArgs& a, int width, float* part, void* out, int out_dt,
                              int64_t out_stride, hipStream_t s) {
    const int tasks = (a.M + 3) / 4 * (a.k / 128);
    hipLaunchKernelGGL(lin_xh_kernel, dim3((unsigned)((tasks + kLxWaves - 1) / kLxWaves)), dim3(64 * kLxWaves), 0, s,
                       (const LinearArgs&)a);
    switch (cb * 8 + K) {
        case 16 + 2: linear_rows_product<2, 2>(a, width, part, out, out_dt, out_stride, s); break;
        case 16 + 3: linear_rows_product<3, 2>(a, width, part, out, out_dt, out_stride, s); break;
        case 16 + 4: linear_rows_product<4, 2>(a, width, part, out, out_dt, out_stride, s); break;
        case 16 + 5: linear_rows_product<5, 2>(a, width, part, out, out_dt, out_stride, s); break;
        case 16 + 6: linear_rows_product<6, 2>(a, width, part, out, out_dt, out_stride, s); break;
        case 8 + 4: linear_rows_product<4, 1>(a, width, part, out, out_dt, out_stride, s); break;
        case 8 + 6: linear_rows_product<6, 1>(a, width, part, out, out_dt, out_stride, s); break;
        case 4: linear_rows_product<4, 0>(a, width, part, out, out_dt, out_stride, s); break;
        case 6: linear_rows_product<6, 0>(a, width, part, out, out_dt, out_stride, s); break;
        default: return hipErrorInvalidValue;
    }
    if (a.P > 1) return launch_linear_had_out(part, 0, a.P, a.M, a.n, a.svh, out, out_dt, out_stride, s);
    return hipGetLastError();
}

}  // namespace exl3
