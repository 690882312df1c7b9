// The two products of the grouped experts (moe_grouped.hip): kernels and their launches for one bitrate K. Each bitrate is
// a translation unit of its own (moe_products_k2.hip, ...).
#pragma once
#include "exl3_common.cuh"
#include "exl3_fill.cuh"
#include "exl3_geom.h"
#include "exl3_kernels.h"
#include "exl3_regb.cuh"

#include <algorithm>

namespace exl3 {

template <int NB> constexpr int kMoePf = NB >= 5 && NB <= 8 ? 4 : 0;
constexpr int kMoeSd = 1;                        // chunks of A in flight in registers (the accumulators leave no room)
constexpr int kEpRow = 260;                      // floats per row of the [16][256] epilogue tile (16-byte reads of 4 rows
                                                 // fall on distinct banks)

// ---- the two products ----------------------------------------------------------------------------------------------------

// wave-uniform values that the compiler loads per lane, as scalars: a descriptor in vector registers would make every
// buffer load a loop over its lanes
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ const uint8_t* item_blob(const GroupedArgs& A, int a) {
    const uint64_t p = (uint64_t)A.it_blob[a];
    return (const uint8_t*)(((uint64_t)(uint32_t)uni((int)(p >> 32)) << 32) | (uint32_t)uni((int)p));
}

// block index -> (item, column block): the nblk workgroups of an item share blockIdx % 8, i.e. one XCD and its L2
__device__ __forceinline__ void gr_block(int blk, int nblk, int& a, int& nb) {
    const int xcd = blk & 7, slot = blk >> 3;
    a = (slot / nblk) * 8 + xcd;
    nb = slot % nblk;
}

// the wave's 64 columns of row block b into its epilogue tile of ROW floats per row
template <int K, int ROW = kEpRow>
__device__ __forceinline__ void stash(const float4_t (&acc)[2][2], float* ep, int wc) {
    using B = RegB<K, false, 2>;
    const int q4 = 4 * (lane_id() >> 4);
#pragma unroll
    for (int cc = 0; cc < 2; ++cc)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int c = wc * 64 + B::col(cc, h);
#pragma unroll
            for (int v = 0; v < 4; ++v) ep[(q4 + v) * ROW + c] = acc[cc][h][v];
        }
}

// 8 outputs of a pick: v * sc * svh, as fp32 or fp16
template <typename TY>
__device__ __forceinline__ void st_y(void* y, size_t o, const float (&v)[8], float sc, const half8_u& hs) {
    if constexpr (sizeof(TY) == 4) {
#pragma unroll
        for (int j = 0; j < 8; j += 4)
            *(float4_t*)((float*)y + o + j) = float4_t{v[j] * sc * (float)hs[j], v[j + 1] * sc * (float)hs[j + 1],
                                                       v[j + 2] * sc * (float)hs[j + 2], v[j + 3] * sc * (float)hs[j + 3]};
    } else {
        half8_t r;
#pragma unroll
        for (int j = 0; j < 8; ++j) r[j] = to_half(v[j] * sc * (float)hs[j]);
        *(half8_t*)((half_t*)y + o) = r;
    }
}

// an item of one block: 4 waves of 64 columns (128 of I, both projections) in each of KS K-slices
template <int K, int KS>
__device__ __forceinline__ void gateup_item(const GroupedArgs& A, int a, int s0, int rows, int nb, float* ep) {
    constexpr int NB = 1;
    const int I = A.g.I, H = A.g.H, tiles_n = 2 * I / 16, l = lane_id();
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wc = wv & 3, ks = wv >> 2, pj = wc >> 1;
    using B = RegB<K, false, 2>;
    const uint8_t* base = item_blob(A, a);
    const auto rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(base), (short)0, (int)A.g.gu_bytes, 0x00020000);
    const auto ra = __builtin_amdgcn_make_buffer_rsrc(A.xh, (short)0, A.npairs * 4 * H, 0x00020000);
    uint32_t aoff[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const int m = 16 * b + (l & 15);
        aoff[b] = m < rows ? (uint32_t)(A.perm[s0 + m] * 2 + pj) * 2u * H + B::a_lane_off() : kOob;
    }
    const uint32_t woff = B::lane_off(tiles_n, pj * (I / 16) + nb * 8 + (wc & 1) * 4);
    const int nch = H / 64;
    float4_t acc[NB][2][2];
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[b][0][0] = acc[b][0][1] = acc[b][1][0] = acc[b][1][1] = float4_t{};
    regb_core<K, NB, false, 2>(rw, woff, tiles_n, ra, aoff, nch * ks / KS, nch * (ks + 1) / KS, acc);
    const int cb8 = nb * 128 + (l & 15) * 8;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        stash<K>(acc[b], ep + ks * 16 * kEpRow, wc);
        __syncthreads();
        if (wv < 4) {                            // 4 rows per wave, 16 lanes x 8 columns per row
            const int rr = wv * 4 + (l >> 4), row = 16 * b + rr;
            const half8_u hg = ld_half8(base + A.g.off_svh_g + 2 * cb8);
            const half8_u hu = ld_half8(base + A.g.off_svh_u + 2 * cb8);
            const half8_u hd = ld_half8(base + A.g.off_suh_d + 2 * cb8);
            float g[8], u[8], av[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) g[j] = u[j] = 0.f;
#pragma unroll
            for (int k = 0; k < KS; ++k) {       // the K-slices in order
                const float* er = ep + (k * 16 + rr) * kEpRow + (l & 15) * 8;
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    g[j] += er[j];
                    u[j] += er[128 + j];
                }
            }
            row_fwht128_signed(g);
            row_fwht128_signed(u);
            const float rs = row_sign() * kRsqrt128;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float gj = (float)to_half(g[j] * rs * (float)hg[j]);
                const float uj = (float)to_half(u[j] * rs * (float)hu[j]);
                const float aj = (float)to_half(silu_mul(gj, uj));
                av[j] = (float)to_half(aj * (float)hd[j]);
            }
            row_fwht128_signed(av);
            half8_t o;
#pragma unroll
            for (int j = 0; j < 8; ++j) o[j] = to_half(av[j] * rs);
            if (row < rows) *(half8_t*)(A.abuf + (size_t)A.perm[s0 + row] * I + cb8) = o;
        }
        if (b + 1 < NB) __syncthreads();
    }
}

// ---- the same with the rows staged in LDS: items of several blocks ----------------------------------------------------
// WV waves of 64 columns: gate/up takes 32 WV columns of I of both projections, down 64 WV columns of H
template <int WV> constexpr int kEpRowW = 64 * WV + 4;

template <int K, int NB, int WV>
__device__ __forceinline__ void gateup_rows(const GroupedArgs& A, int a, int s0, int rows, int nb, uint8_t* lds) {
    const int I = A.g.I, H = A.g.H, tiles_n = 2 * I / 16, l = lane_id();
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int pj = wv / (WV / 2), wc = wv % (WV / 2);
    using B = RegB<K, false, 2>;
    using U = AUnits<NB, WV, 2>;
    const uint8_t* base = item_blob(A, a);
    const auto rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(base), (short)0, (int)A.g.gu_bytes, 0x00020000);
    const auto ra = __builtin_amdgcn_make_buffer_rsrc(A.xh, (short)0, A.npairs * 4 * H, 0x00020000);
    uint32_t soff[U::NU];
#pragma unroll
    for (int i = 0; i < U::NU; ++i) {
        const int m = U::row(i);
        soff[i] = U::live(i) && m < rows ? (uint32_t)(A.perm[s0 + m] * 2 + U::proj(i)) * 2u * H + 32u * (U::index(i) & 3)
                                         : kOob;
    }
    float4_t acc[NB][2][2];
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[b][0][0] = acc[b][0][1] = acc[b][1][0] = acc[b][1][1] = float4_t{};
    regb_lds_core<K, NB, WV, 2, false, 2, kMoeSd, kMoePf<NB>>(
        rw, B::lane_off(tiles_n, pj * (I / 16) + nb * 2 * WV + wc * 4), tiles_n, ra, soff, H / 64, pj, lds, acc);
    // 16 rows per round through one of two tiles [16][gate 32 WV | up 32 WV]: 16 lanes per (row, 128 columns)
    const int un = threadIdx.x >> 4, rr = un & 15, cb = (un >> 4) * 128 + (l & 15) * 8, ci = nb * 32 * WV + cb;
    const half8_u hg = ld_half8(base + A.g.off_svh_g + 2 * ci);
    const half8_u hu = ld_half8(base + A.g.off_svh_u + 2 * ci);
    const half8_u hd = ld_half8(base + A.g.off_suh_d + 2 * ci);
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        float* ep = (float*)lds + (b & 1) * 16 * kEpRowW<WV>;
        stash<K, kEpRowW<WV>>(acc[b], ep, wv);
        __syncthreads();
        const float* er = ep + rr * kEpRowW<WV> + cb;
        float g[8], u[8], av[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            g[j] = er[j];
            u[j] = er[32 * WV + j];
        }
        row_fwht128_signed(g);
        row_fwht128_signed(u);
        const float rs = row_sign() * kRsqrt128;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float gj = (float)to_half(g[j] * rs * (float)hg[j]);
            const float uj = (float)to_half(u[j] * rs * (float)hu[j]);
            const float aj = (float)to_half(silu_mul(gj, uj));
            av[j] = (float)to_half(aj * (float)hd[j]);
        }
        row_fwht128_signed(av);
        half8_t o;
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = to_half(av[j] * rs);
        const int row = 16 * b + rr;
        if (row < rows) *(half8_t*)(A.abuf + (size_t)A.perm[s0 + row] * I + ci) = o;
    }
}

// (LDSA: A staged through LDS, else each wave's own loads)
template <int K, int NB, int WV, bool LDSA, typename TY>
__device__ __forceinline__ void down_rows(const GroupedArgs& A, int a, int s0, int rows, int nt, uint8_t* lds) {
    const int I = A.g.I, H = A.g.H, tiles_n = H / 16, l = lane_id();
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    using B = RegB<K, false, 2>;
    using U = AUnits<NB, WV, 1>;
    const uint8_t* base = item_blob(A, a);
    const auto rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(base) + A.g.gu_bytes, (short)0,
                                                      (int)A.g.d_bytes, 0x00020000);
    const auto ra = __builtin_amdgcn_make_buffer_rsrc(A.abuf, (short)0, A.npairs * 2 * I, 0x00020000);
    float4_t acc[NB][2][2];
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[b][0][0] = acc[b][0][1] = acc[b][1][0] = acc[b][1][1] = float4_t{};
    const uint32_t woff = B::lane_off(tiles_n, nt * 4 * WV + wv * 4);
    if constexpr (LDSA) {
        uint32_t soff[U::NU];
#pragma unroll
        for (int i = 0; i < U::NU; ++i) {
            const int m = U::row(i);
            soff[i] = U::live(i) && m < rows ? (uint32_t)A.perm[s0 + m] * 2u * I + 32u * (U::index(i) & 3) : kOob;
        }
        regb_lds_core<K, NB, WV, 1, false, 2, kMoeSd, kMoePf<NB>>(rw, woff, tiles_n, ra, soff, I / 64, 0, lds, acc);
    } else {
        uint32_t aoff[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int m = 16 * b + (l & 15);
            aoff[b] = m < rows ? (uint32_t)A.perm[s0 + m] * 2u * I + B::a_lane_off() : kOob;
        }
        regb_core<K, NB, false, 2>(rw, woff, tiles_n, ra, aoff, 0, I / 64, acc);
    }
    // 16 rows per round, 16 lanes per (row, 128 columns), two units per thread. The output scales are loaded once: per
    // round, the 16 rows of an expert in host memory read as many bytes of them over PCIe as 40 % of its trellis
    half8_u hs[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
        hs[i] = ld_half8(base + A.g.off_svh_d +
                         2 * (nt * 64 * WV + (((int)(threadIdx.x >> 4) + i * 4 * WV) >> 4) * 128 + (l & 15) * 8));
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        float* ep = (float*)lds + (b & 1) * 16 * kEpRowW<WV>;
        stash<K, kEpRowW<WV>>(acc[b], ep, wv);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int un = (threadIdx.x >> 4) + i * 4 * WV, rr = un & 15, cb = (un >> 4) * 128 + (l & 15) * 8;
            const int row = 16 * b + rr, ch = nt * 64 * WV + cb;
            const int pk = A.perm[s0 + min(row, rows - 1)];
            const float pw = A.w[pk];
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = ep[rr * kEpRowW<WV> + cb + j];
            row_fwht128_signed(v);
            if (row < rows) st_y<TY>(A.y, (size_t)pk * H + ch, v, row_sign() * kRsqrt128 * pw, hs[i]);
        }
    }
}

// an item of one block: 4 waves of 64 columns (256 of H) in each of KS K-slices
template <int K, int KS, typename TY>
__device__ __forceinline__ void down_item(const GroupedArgs& A, int a, int s0, int rows, int nt, float* ep) {
    const int I = A.g.I, H = A.g.H, tiles_n = H / 16, l = lane_id();
    const int wv = uni(threadIdx.x >> 6), wc = wv & 3, ks = wv >> 2;
    using B = RegB<K, false, 2>;
    const uint8_t* base = item_blob(A, a);
    const auto rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(base) + A.g.gu_bytes, (short)0,
                                                      (int)A.g.d_bytes, 0x00020000);
    const auto ra = __builtin_amdgcn_make_buffer_rsrc(A.abuf, (short)0, A.npairs * 2 * I, 0x00020000);
    const int m = l & 15;
    const uint32_t aoff[1] = {m < rows ? (uint32_t)A.perm[s0 + m] * 2u * I + B::a_lane_off() : kOob};
    float4_t acc[1][2][2];
    acc[0][0][0] = acc[0][0][1] = acc[0][1][0] = acc[0][1][1] = float4_t{};
    const int nch = I / 64;
    regb_core<K, 1, false, 2>(rw, B::lane_off(tiles_n, nt * 16 + wc * 4), tiles_n, ra, aoff, nch * ks / KS,
                              nch * (ks + 1) / KS, acc);
    stash<K>(acc[0], ep + ks * 16 * kEpRow, wc);
    __syncthreads();
    // 16 rows x 2 halves of 128 columns, 16 lanes each
#pragma unroll
    for (int u0 = 0; u0 < 32; u0 += 16 * KS) {
        const int un = u0 + (threadIdx.x >> 4), rr = un & 15, cb = (un >> 4) * 128 + (l & 15) * 8, ch = nt * 256 + cb;
        const int pk = A.perm[s0 + min(rr, rows - 1)];
        const half8_u hs = ld_half8(base + A.g.off_svh_d + 2 * ch);
        const float pw = A.w[pk];
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = 0.f;
#pragma unroll
        for (int k = 0; k < KS; ++k)             // the K-slices in order
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] += ep[(k * 16 + rr) * kEpRow + cb + j];
        row_fwht128_signed(v);
        if (rr < rows) st_y<TY>(A.y, (size_t)pk * H + ch, v, row_sign() * kRsqrt128 * pw, hs);
    }
}

// One launch per product (two launches, one per item size, left the chip idle behind the longest item of each: a batch
// of 64 rows took 193 us in two, 132 us in one). !BIG (items of up to 4 blocks): 4 waves per SIMD; the items of several
// blocks come first, then those of one. BIG (items of up to 12 blocks): 2 waves per SIMD, block counts below 9 rounded up
// to 4, 6 or 8. A kernel holds up to seven instantiations of the core, and its largest sets the registers of all: at 128 and
// 256 VGPRs the compiler spills 4-10 of them at K = 3, 8-31 at K = 4 (most in the 4-wave gate/up).
// FILL: the instantiations that copy (exl3_fill.cuh); the copy inside the others would cost them up to 3 % in registers.
template <int K, int WV, bool BIG, bool FILL>
__global__ void __launch_bounds__(64 * WV) __attribute__((amdgpu_waves_per_eu(BIG ? 2 : 4)))
grouped_gateup_kernel(GroupedArgs A) {
    constexpr int kLds = std::max(2 * AUnits<BIG ? 12 : 4, WV, 2>::kBuf, 2 * 16 * kEpRowW<WV> * 4);
    __shared__ __align__(16) uint8_t lds[kLds];
    int blk = blockIdx.x, a, nb;
    if constexpr (FILL) {                        // a cached call's misses: their down trellis
        if (blk < fill_workgroups(64 * WV)) {
            fill_part<64 * WV>(A, 1, blk);
            return;
        }
        blk -= fill_workgroups(64 * WV);
    }
    const int nblk = A.g.I / (32 * WV), nmany = uni(A.n_items[BIG ? 0 : 1]);
    const int bmany = (nmany + 7) / 8 * 8 * nblk;
    if (BIG || blk < bmany) {
        gr_block(blk, nblk, a, nb);
        if (a >= nmany) return;
    } else {
        if constexpr (!BIG) {
            gr_block(blk - bmany, A.g.I / 128, a, nb);
            a += nmany;
            if (a >= A.n_items[0]) return;
            gateup_item<K, WV / 4>(A, a, uni(A.it_start[a]), uni(A.it_cnt[a]), nb, (float*)lds);
        }
        return;
    }
    const int s0 = uni(A.it_start[a]), rows = uni(A.it_cnt[a]), bl = (rows + 15) >> 4;
    if constexpr (!BIG) {
        if (bl <= 2) gateup_rows<K, 2, WV>(A, a, s0, rows, nb, lds);
        else if (bl == 3) gateup_rows<K, 3, WV>(A, a, s0, rows, nb, lds);
        else gateup_rows<K, 4, WV>(A, a, s0, rows, nb, lds);
    } else {
        if (bl <= 4) gateup_rows<K, 4, WV>(A, a, s0, rows, nb, lds);
        else if (bl <= 6) gateup_rows<K, 6, WV>(A, a, s0, rows, nb, lds);
        else if (bl <= 8) gateup_rows<K, 8, WV>(A, a, s0, rows, nb, lds);
        else if (bl == 9) gateup_rows<K, 9, WV>(A, a, s0, rows, nb, lds);
        else if (bl == 10) gateup_rows<K, 10, WV>(A, a, s0, rows, nb, lds);
        else if (bl == 11) gateup_rows<K, 11, WV>(A, a, s0, rows, nb, lds);
        else gateup_rows<K, 12, WV>(A, a, s0, rows, nb, lds);
    }
}

template <int K, int WV, bool BIG, typename TY>
__global__ void __launch_bounds__(64 * WV) __attribute__((amdgpu_waves_per_eu(BIG ? 2 : 4)))
grouped_down_kernel(GroupedArgs A) {
    constexpr int kLds = std::max(2 * AUnits<BIG ? 12 : 4, WV, 1>::kBuf, 2 * 16 * kEpRowW<WV> * 4);
    __shared__ __align__(16) uint8_t lds[kLds];
    // the items of one block apart, at the decode sizes (fp32 outputs): there are few, and 256 columns x 2 K-slices spread
    // them better than 512 columns (16 rows 23 -> 19 us, 6 rows of wide experts 62 -> 45 us); 512 experts of 5 rows fill
    // the chip either way and take 97 us in 512 columns against 99
    constexpr bool kOne = !BIG && sizeof(TY) == 4;
    const int nblk = A.g.H / (64 * WV), nmany = uni(A.n_items[kOne ? 1 : 0]);
    const int blk = blockIdx.x, bmany = (nmany + 7) / 8 * 8 * nblk;
    int a, nt;
    if (!kOne || blk < bmany) {
        gr_block(blk, nblk, a, nt);
        if (a >= nmany) return;
    } else {
        if constexpr (kOne) {
            gr_block(blk - bmany, A.g.H / 256, a, nt);
            a += nmany;
            if (a >= uni(A.n_items[0])) return;
            down_item<K, WV / 4, TY>(A, a, uni(A.it_start[a]), uni(A.it_cnt[a]), nt, (float*)lds);
        }
        return;
    }
    const int s0 = uni(A.it_start[a]), rows = uni(A.it_cnt[a]), bl = (rows + 15) >> 4;
    if constexpr (!BIG) {
        if (!kOne && bl == 1) down_rows<K, 1, WV, false, TY>(A, a, s0, rows, nt, lds);
        else if (bl <= 2) down_rows<K, 2, WV, true, TY>(A, a, s0, rows, nt, lds);
        else if (bl == 3) down_rows<K, 3, WV, true, TY>(A, a, s0, rows, nt, lds);
        else down_rows<K, 4, WV, true, TY>(A, a, s0, rows, nt, lds);
    } else {
        if (bl <= 4) down_rows<K, 4, WV, true, TY>(A, a, s0, rows, nt, lds);
        else if (bl <= 6) down_rows<K, 6, WV, true, TY>(A, a, s0, rows, nt, lds);
        else if (bl <= 8) down_rows<K, 8, WV, true, TY>(A, a, s0, rows, nt, lds);
        else if (bl == 9) down_rows<K, 9, WV, true, TY>(A, a, s0, rows, nt, lds);
        else if (bl == 10) down_rows<K, 10, WV, true, TY>(A, a, s0, rows, nt, lds);
        else if (bl == 11) down_rows<K, 11, WV, true, TY>(A, a, s0, rows, nt, lds);
        else down_rows<K, 12, WV, true, TY>(A, a, s0, rows, nt, lds);
    }
}

template <int K>
void launch_products(const GroupedArgs& a, bool y32, hipStream_t s) {
    const size_t np = a.npairs, mi = grouped_max_items(np, a.E);
    auto g8 = [](size_t items) { return (unsigned)((items + 7) / 8 * 8); };
    const int I = a.g.I, H = a.g.H;
    const bool big = a.rmax > 64;                // (8-wave layouts and fp16 outputs only, moe_grouped.hip)
    auto run = [&](auto kern, unsigned grid, int nt) { hipLaunchKernelGGL(kern, dim3(grid), dim3(nt), 0, s, a); };
    GroupedArgs b = a;                           // the experts of more than 64 rows, where they are listed apart
    b.it_blob = a.big_blob;
    b.it_start = a.big_start;
    b.it_cnt = a.big_cnt;
    b.n_items = a.big_n;
    auto apart = [&](auto kern, int blocks) {
        if (a.big_n && np > 64) hipLaunchKernelGGL(kern, dim3(g8(np / 65) * blocks), dim3(512), 0, s, b);
    };
    apart(grouped_gateup_kernel<K, 8, true, false>, I / 256);
    // items of several blocks hold at least 17 rows each
    const unsigned many = g8(np / 17), one = g8(std::min<size_t>(np, a.E));
    if (big) {
        run(grouped_gateup_kernel<K, 8, true, false>, g8(mi) * (I / 256), 512);
    } else if (I % 256 == 0) {
        const unsigned grid = many * (I / 256) + one * (I / 128);
        if (a.f.list) run(grouped_gateup_kernel<K, 8, false, true>, fill_workgroups(512) + grid, 512);
        else run(grouped_gateup_kernel<K, 8, false, false>, grid, 512);
    } else {
        const unsigned grid = (many + one) * (I / 128);
        if (a.f.list) run(grouped_gateup_kernel<K, 4, false, true>, fill_workgroups(256) + grid, 256);
        else run(grouped_gateup_kernel<K, 4, false, false>, grid, 256);
    }
    apart(grouped_down_kernel<K, 8, true, half_t>, H / 512);
    auto down = [&](auto ty) {
        using TY = decltype(ty);
        const unsigned ones = one * (H / 256);
        if (H % 512 == 0) run(grouped_down_kernel<K, 8, false, TY>, y32 ? many * (H / 512) + ones : g8(mi) * (H / 512), 512);
        else run(grouped_down_kernel<K, 4, false, TY>, y32 ? many * (H / 256) + ones : g8(mi) * (H / 256), 256);
    };
    if (big) run(grouped_down_kernel<K, 8, true, half_t>, g8(mi) * (H / 512), 512);
    else if (y32) down(float{});
    else down(half_t{});
}

}  // namespace exl3
