// The dense EXL3 linear for more rows than the fused small path takes: out[M, n] = svh * H(sum_k xh[shard of n][m][k]
// W[k][n]) / sqrt 128 with the trellis decoded into MFMA B registers (exl3_regb.cuh), so the weights are never written
// to memory (reference: experimental/n111-victim-ring/csrc/exl3_ops.sycl:651-757; HadInKernel / HadOutKernel,
// exl3_esimd.h:286-343).
//
//   xh    input Hadamards of every (shard, row) as MFMA products with H128, fp16
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

#include <algorithm>

namespace exl3 {

typedef float float16_t __attribute__((ext_vector_type(16)));
typedef _Float16 half8_u __attribute__((ext_vector_type(8), aligned(2)));   // activations and scales at any alignment
typedef float float4_u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x4_u __attribute__((ext_vector_type(4), aligned(2)));

// ---- input Hadamards: one wave per (32 rows, 128-block), every shard -----------------------------------------------------
constexpr int kLxWaves = 8;
constexpr int kLxRow = 64 + 8;                   // LDS row of one row's half block (halfs, padded)

template <int DT>
__device__ __forceinline__ void lx_load(const void* x, size_t i, float (&v)[8]) {
    if constexpr (DT == 2) {
        const float4_u a = *(const float4_u*)((const float*)x + i), b = *(const float4_u*)((const float*)x + i + 4);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            v[j] = a[j];
            v[4 + j] = b[j];
        }
    } else if constexpr (DT == 1) {
        const u32x4_u w = *(const u32x4_u*)((const bf16_bits*)x + i);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            v[2 * j] = __uint_as_float(w[j] << 16);
            v[2 * j + 1] = __uint_as_float(w[j] & 0xFFFF0000u);
        }
    } else {
        const half8_u h = *(const half8_u*)((const half_t*)x + i);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = (float)h[j];
    }
}

template <int DT>
__device__ __forceinline__ void lx_task(const LinearArgs& A, int g, int rb, int kb, half_t* tb) {
    const int l = lane_id();
    half8_t hf[2][2];                            // [ks & 1][negated]: rows n' = l % 32, k' = 8 (l / 32) + j of H
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const bool neg = __popc((l & 31) & (b * 16 + (l >> 5) * 8 + j)) & 1;
            hf[b][0][j] = neg ? (half_t)-1.0f : (half_t)1.0f;
            hf[b][1][j] = neg ? (half_t)1.0f : (half_t)-1.0f;
        }
    const int m0 = rb * 32;
    const size_t xrow = (size_t)min(m0 + (l & 31), A.M - 1) * A.x_stride;
    const half_t* su = A.suh + (size_t)g * A.k;
    half8_t bx[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int kk = kb * 128 + i * 16 + (l >> 5) * 8;
        float xv[8];
        lx_load<DT>(A.x, xrow + kk, xv);
        const half8_u sv = *(const half8_u*)(su + kk);
#pragma unroll
        for (int j = 0; j < 8; ++j) bx[i][j] = to_half(xv[j] * (float)sv[j]);
    }
#pragma unroll
    for (int hb = 0; hb < 2; ++hb) {
#pragma unroll
        for (int n2 = 0; n2 < 2; ++n2) {
            const int nb = 2 * hb + n2;
            float16_t acc = float16_t{};
#pragma unroll
            for (int i = 0; i < 8; ++i)
                acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(hf[i & 1][__popc(nb & (i >> 1)) & 1], bx[i], acc, 0, 0, 0);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
                *(half4_t*)(tb + (l & 31) * kLxRow + n2 * 32 + q * 8 + (l >> 5) * 4) =
                    half4_t{to_half(acc[4 * q] * kRsqrt128), to_half(acc[4 * q + 1] * kRsqrt128),
                            to_half(acc[4 * q + 2] * kRsqrt128), to_half(acc[4 * q + 3] * kRsqrt128)};
            }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {            // the wave's own LDS rows: 8 rows x 128 bytes per store
            const int pr = r * 8 + (l >> 3), col = (l & 7) * 8;
            const half8_t v = *(const half8_t*)(tb + pr * kLxRow + col);
            if (m0 + pr < A.M) *(half8_t*)(A.xh + ((size_t)g * A.M + m0 + pr) * A.k + kb * 128 + hb * 64 + col) = v;
        }
    }
}

__global__ void __launch_bounds__(64 * kLxWaves) lin_xh_kernel(LinearArgs A) {
    __shared__ __align__(16) half_t tbuf[kLxWaves][32 * kLxRow];
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kbn = A.k / 128, t = blockIdx.x * kLxWaves + wv, nrb = (A.M + 31) / 32;
    if (t >= A.S * nrb * kbn) return;
    const int kb = t % kbn, g = (t / kbn) % A.S, rb = t / (kbn * A.S);   // the shards of a block share x in L2
    if (A.x_dt == 1) lx_task<1>(A, g, rb, kb, tbuf[wv]);
    else if (A.x_dt == 2) lx_task<2>(A, g, rb, kb, tbuf[wv]);
    else lx_task<0>(A, g, rb, kb, tbuf[wv]);
}

// ---- host --------------------------------------------------------------------------------------------------------------

int linear_rows_slices(int M, int k, int n, int width) {
    const int rt = 16 * linear_rows_blocks(M), wgs = (n / width) * ((M + rt - 1) / rt), nkb = k / 128;
    // about one workgroup of 8 waves per CU: more slices cost their partial sums' traffic (40 rows, 2048 -> 12,288, K 4,
    // 48 workgroups: 1 / 2 / 4 / 8 slices 37 / 29 / 26 / 34 us; 1,024 rows, 4096 -> 2048, 64 workgroups: 84 / 58 / 48 /
    // 61 us), and up to 512 input rows a second launch for the sums costs more than the slices give (1,024 rows, 512 ->
    // 2048: 25 against 31 us)
    return nkb <= 4 ? 1 : std::max(1, std::min(std::min(8, nkb / 2), 256 / wgs));
}

hipError_t launch_linear_rows(int K, int cb, const LinearArgs& a, int width, float* part, void* out, int out_dt,
                              int64_t out_stride, hipStream_t s) {
    const int tasks = a.S * ((a.M + 31) / 32) * (a.k / 128);
    hipLaunchKernelGGL(lin_xh_kernel, dim3((unsigned)((tasks + kLxWaves - 1) / kLxWaves)), dim3(64 * kLxWaves), 0, s, a);
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
