// The product of the dense linear for more rows (linear_rows.hip) and its launch for one bitrate and codebook; a few of
// these to a translation unit (linear_rows_k23.hip, ...).
#pragma once
#include "exl3_common.cuh"
#include "exl3_kernels.h"
#include "exl3_regb.cuh"

#include <algorithm>

namespace exl3 {

// A workgroup of 2 CW waves: CW waves of 64 columns for each half of its K-slice (twice the waves per SIMD that the
// columns alone give, at no traffic: the halves are summed in LDS). Each half is staged as a matrix of its own.
template <int K, int CB, int NB, int CW>
__global__ void __launch_bounds__(128 * CW) __attribute__((amdgpu_waves_per_eu(NB <= 2 ? 4 : NB <= 4 ? 3 : 2)))
lin_rows_kernel(LinearRowsArgs A, float* part, void* out, int out_dt, int64_t out_stride, int vec) {
    constexpr int WV = 2 * CW;
    using B = RegB<K, true, CB>;
    using U = AUnits<NB, WV, 2>;
    constexpr int kRow = 64 * CW + 4;            // floats per row of an epilogue tile [16][64 CW]
    constexpr int kTile = 16 * kRow;
    __shared__ __align__(16) uint8_t lds[std::max(2 * U::kBuf, 4 * kTile * 4)];
    const int ntile = A.n / (64 * CW), l = lane_id();
    const int ct = blockIdx.x % ntile, ks = (blockIdx.x / ntile) % A.P, m0 = blockIdx.x / (ntile * A.P) * 16 * NB;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wc = wv % CW, kh = wv / CW;
    const int n0 = ct * 64 * CW, nkb = A.k / 128, b0 = nkb * ks / A.P, half = nkb * (ks + 1) / A.P - b0;
    const int c0 = 2 * b0;                       // the slice's first chunk; each half of it has `half` chunks
    int g = 0;                                   // one shard per workgroup (the tile width divides the bounds)
    for (int j = 1; j < A.S; ++j) g = n0 >= A.first[j] ? j : g;
    const auto rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(A.tr), (short)0,
                                                      (int)((int64_t)A.k * A.n / 8 * K), 0x00020000);
    const auto ra = __builtin_amdgcn_make_buffer_rsrc(A.xh, (short)0, (int)((int64_t)A.S * A.M * A.k * 2), 0x00020000);
    uint32_t soff[U::NU];
#pragma unroll
    for (int i = 0; i < U::NU; ++i) {
        const int m = m0 + U::row(i);
        soff[i] = U::live(i) && m < A.M
                      ? (uint32_t)(g * A.M + m) * 2u * A.k + 32u * (U::index(i) & 3) + 128u * (c0 + U::proj(i) * half) : kOob;
    }
    float4_t acc[NB][2][2];
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[b][0][0] = acc[b][0][1] = acc[b][1][0] = acc[b][1][1] = float4_t{};
    const uint32_t woff = B::lane_off(A.n / 16, n0 / 16 + wc * 4) + (uint32_t)(c0 + kh * half) * B::chunk_bytes(A.n / 16);
    regb_lds_core<K, NB, WV, 2, true, CB, NB <= 4 ? 2 : 1, NB <= 4 ? 0 : 4>(rw, woff, A.n / 16, ra, soff, half, kh, lds, acc);
    // 16 rows per round through one of two pairs of tiles, 16 lanes per (row, 128 columns)
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        float* ep = (float*)lds + (b & 1) * 2 * kTile;
        const int q4 = 4 * (l >> 4);
#pragma unroll
        for (int cc = 0; cc < 2; ++cc)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    ep[kh * kTile + (q4 + v) * kRow + wc * 64 + B::col(cc, h)] = acc[b][cc][h][v];
        __syncthreads();
        const int un = threadIdx.x >> 4, rr = un & 15, cb = (un >> 4) * 128 + (l & 15) * 8;
        const int row = m0 + 16 * b + rr, col = n0 + cb;
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = ep[rr * kRow + cb + j] + ep[kTile + rr * kRow + cb + j];
        if (A.P > 1) {
            if (row < A.M) {
                float* p = part + ((size_t)ks * A.M + row) * A.n + col;
                *(float4_t*)p = float4_t{v[0], v[1], v[2], v[3]};
                *(float4_t*)(p + 4) = float4_t{v[4], v[5], v[6], v[7]};
            }
            continue;
        }
        row_fwht128_signed(v);
        const half8_u sv = *(const half8_u*)(A.svh + col);
        const float rs = row_sign() * kRsqrt128;
        if (row < A.M) {
            const size_t o = (size_t)row * out_stride + col;
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = v[j] * rs * (float)sv[j];
            if (vec && out_dt != 2) {            // 16-bit outputs whose rows start on 16 bytes
                u32x4_t w;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    w[j] = out_dt == 1 ? (uint32_t)f32_to_bf16(v[2 * j]) | ((uint32_t)f32_to_bf16(v[2 * j + 1]) << 16)
                                       : (uint32_t)__builtin_bit_cast(uint16_t, to_half(v[2 * j])) |
                                             ((uint32_t)__builtin_bit_cast(uint16_t, to_half(v[2 * j + 1])) << 16);
                *(u32x4_t*)((uint16_t*)out + o) = w;
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) st_act(out, out_dt, o + j, v[j]);
            }
        }
    }
}

template <int K, int CB>
void linear_rows_product(const LinearRowsArgs& a, int width, float* part, void* out, int out_dt, int64_t out_stride,
                        hipStream_t s) {
    const int nb = linear_rows_blocks(a.M), vec = (out_stride & 7) == 0 && ((uintptr_t)out & 15) == 0;
    const dim3 grid((unsigned)((a.n / width) * a.P * ((a.M + 16 * nb - 1) / (16 * nb))));
    auto run = [&](auto kern, int nt) { hipLaunchKernelGGL(kern, grid, dim3(nt), 0, s, a, part, out, out_dt, out_stride, vec); };
    if (width == 256) {
        if (nb == 1) run(lin_rows_kernel<K, CB, 1, 4>, 512);
        else if (nb == 2) run(lin_rows_kernel<K, CB, 2, 4>, 512);
        else if (nb == 4) run(lin_rows_kernel<K, CB, 4, 4>, 512);
        else run(lin_rows_kernel<K, CB, 8, 4>, 512);
    } else {
        if (nb == 1) run(lin_rows_kernel<K, CB, 1, 2>, 256);
        else if (nb == 2) run(lin_rows_kernel<K, CB, 2, 2>, 256);
        else if (nb == 4) run(lin_rows_kernel<K, CB, 4, 2>, 256);
        else run(lin_rows_kernel<K, CB, 8, 2>, 256);
    }
}

}  // namespace exl3
