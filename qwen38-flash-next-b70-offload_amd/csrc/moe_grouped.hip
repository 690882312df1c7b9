// Routed experts with the picks grouped by expert (decode batches and prompts): every expert's trellis is decoded once
// per item of up to 64 or 192 rows, straight into MFMA B registers (exl3_regb.cuh).
//
//   pre      one launch: workgroup 0 sorts the picks by expert and cuts them into items (longest first), the others
//            write the input Hadamards xh of every (pick, projection), which need no sort
//   gate/up  per (item, 32 WV columns of I), WV waves of 64 columns, half of them on each projection; the rows gathered
//            by pick; epilogue through LDS: g/u Hadamards, SwiGLU, * suh_d, Hadamard -> abuf[pick] (fp16)
//   down     per (item, 64 WV columns of H), K = I, the same core; output Hadamard * (w * svh_d) -> y[pick]
//   combine  out[m] = sum over the row's picks of y, in pick order (fp32)
// (reference: kernels/moe-a8/exl3_moe.a8.sycl:121-395, 422-635, 639-680, with the same fp16 rounding points.)
//
// What bounds them: the decode's VALU work, 3.5 instructions per weight (bfe, mul_lo, sad, half a pk_fma) at 4.2 to 4.6
// clocks each per wave of 64. At H 2048 / I 512 / K 3 with all 512 experts active that is 155 us per layer at 2.4 GHz
// against 97 us for the 612 MB of weights at 6.3 TB/s; with up to 16 rows per expert (301 tokens, top-10) gate/up
// takes 150-170 us and down 85-98 us, 89 % and 79 % of their VALU cycles issuing. Columns are split over waves, not K,
// so that a weight is decoded by one wave and multiplied into every row, and nothing is exchanged before the epilogue.
// Whole layers, bf16, before (one decode per pick, or a core that decodes into LDS for 192-row passes) and now:
// 16 Zipf rows 104 -> 74 us, 64 rows 398 -> 132 us, 301 tokens 605 -> 240 us, 2,048 tokens 726 -> 402 us, 8,192 tokens
// 1,290 -> 1,185 us; H 4096 / I 1536, 128 experts, top-8, K 2, 777 tokens: 861 -> 533 us.
#include "exl3_common.cuh"
#include "exl3_geom.h"
#include "exl3_kernels.h"
#include "exl3_regb.cuh"

#include <algorithm>

namespace exl3 {

typedef float float16_t __attribute__((ext_vector_type(16)));

constexpr int kEpRow = 260;                      // floats per row of the [16][256] epilogue tile (16-byte reads of 4 rows
                                                 // fall on distinct banks)
constexpr int kPreThreads = 1024;

// ---- sort into items ---------------------------------------------------------------------------------------------------

__device__ __forceinline__ uint64_t wave_incl_scan64(uint64_t v) {
    const int l = lane_id();
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint64_t t = __shfl_up((unsigned long long)v, d, 64);
        if (l >= d) v += t;
    }
    return v;
}
// exclusive scan over the 1,024 threads of a workgroup; tot = the sum. sw: LDS [17]
__device__ __forceinline__ uint64_t block_scan64(uint64_t v, uint64_t* sw, uint64_t& tot) {
    const int l = lane_id(), w = threadIdx.x >> 6;
    const uint64_t inc = wave_incl_scan64(v);
    if (l == 63) sw[w] = inc;
    __syncthreads();
    if (w == 0) {
        const uint64_t x = l < 16 ? sw[l] : 0;
        const uint64_t xi = wave_incl_scan64(x);
        if (l < 16) sw[l] = xi - x;
        if (l == 15) sw[16] = xi;
    }
    __syncthreads();
    const uint64_t r = sw[w] + inc - v;
    tot = sw[16];
    __syncthreads();
    return r;
}

// thread e: the items of expert e (tot rows from sorted position st): the fewest items of at most rmax rows, cut evenly
// in 16-row blocks; ordered by descending block count over all experts (packed scans of 16 bits per block count), so
// that the longest start first. n_items[0]: all items, [1]: those of more than one block.
constexpr int kMaxBlocks = 12;
__device__ __forceinline__ void emit_items(const GroupedArgs& A, int e, int st, int tot, uint64_t* sw) {
    const int n = (tot + A.rmax - 1) / A.rmax, nb = n ? ((tot + n - 1) / n + 15) >> 4 : 0;   // items, blocks of each
    int above = 0;
    for (int g = (A.rmax + 63) / 64 - 1; g >= 0; --g) {          // block counts 4 g + 1 .. 4 g + 4
        uint64_t tt;
        const uint64_t ex = block_scan64(nb > 4 * g && nb <= 4 * g + 4 ? (uint64_t)n << (16 * (nb - 1 - 4 * g)) : 0ull, sw, tt);
#pragma unroll
        for (int k = 4; k >= 1; --k) {
            if (4 * g + k == nb) {
                int p = above + (int)((ex >> (16 * (k - 1))) & 0xFFFF);
                for (int i = 0; i < n; ++i, ++p) {
                    A.it_expert[p] = e;
                    A.it_start[p] = st + i * 16 * nb;
                    A.it_cnt[p] = min(16 * nb, tot - i * 16 * nb);
                }
            }
            if (g == 0 && k == 1 && threadIdx.x == 0) A.n_items[1] = above;
            above += (int)((tt >> (16 * (k - 1))) & 0xFFFF);
        }
    }
    if (threadIdx.x == 0) A.n_items[0] = above;
}

// the whole sort in one workgroup: counts, starts, items, then the picks' positions. The order of an expert's picks is
// whatever the LDS atomics give: a row's result does not depend on its position (every row of a tile runs the same
// operations on its own data).
__device__ __forceinline__ void sort_wg(const GroupedArgs& A, int* off /* LDS [E] */, uint64_t* sw) {
    const int t = threadIdx.x;
    for (int e = t; e < A.E; e += kPreThreads) off[e] = 0;
    __syncthreads();
    // 8 ids in flight per thread and round
    auto each = [&](auto&& f) {
        for (int i0 = t; i0 < A.npairs; i0 += 8 * kPreThreads) {
            int e[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) e[j] = min(max(A.ids[min(i0 + j * kPreThreads, A.npairs - 1)], 0), A.E - 1);
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (i0 + j * kPreThreads < A.npairs) f(i0 + j * kPreThreads, e[j]);
        }
    };
    each([&](int, int e) { atomicAdd(&off[e], 1); });
    __syncthreads();
    const int tot = t < A.E ? off[t] : 0;
    uint64_t all;
    const int st = (int)block_scan64((uint64_t)tot, sw, all);
    if (t < A.E) off[t] = st;
    emit_items(A, t, st, tot, sw);               // (its barriers order the starts before the positions)
    each([&](int i, int e) { A.perm[atomicAdd(&off[e], 1)] = i; });
}

// ---- input Hadamards ---------------------------------------------------------------------------------------------------
// xh[pick][pj][kb * 128 + n] = fp16(sum_k H[n][k] fp16(x[row][kb * 128 + k] suh_pj[kb * 128 + k]) / sqrt 128) as MFMA
// products C^T = H128 xt^T (A fragments: two per-lane +-1 fragments and their negatives, from the bit split of
// popc(n & k); B = 32 picks). One wave per (32 picks, projection, kbs 128-blocks), results through LDS in halves of 64
// columns, so that 8 lanes store 128 contiguous bytes of a pick.
constexpr int kXhRow = 64 + 8;                   // LDS row of one pick's half block (halfs, padded)
typedef _Float16 half8_u __attribute__((ext_vector_type(8), aligned(2)));   // activations and blob vectors: any alignment
typedef float float4_u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x4_u __attribute__((ext_vector_type(4), aligned(2)));

template <int DT>
__device__ __forceinline__ void ld_x8(const void* x, size_t i, float (&v)[8]) {
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
__device__ __forceinline__ void xh_task(const GroupedArgs& A, int task, int kbs, half_t* tb) {
    const int H = A.g.H, nkb = H / 128, nks = (nkb + kbs - 1) / kbs;
    const int l = lane_id();
    const int pj = task & 1, ks = (task >> 1) % nks, blk = (task >> 1) / nks;
    half8_t hf[2][2];                            // [ks & 1][negated]: rows n' = l % 32, k' = 8 (l / 32) + j
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const bool neg = __popc((l & 31) & (b * 16 + (l >> 5) * 8 + j)) & 1;
            hf[b][0][j] = neg ? (half_t)-1.0f : (half_t)1.0f;
            hf[b][1][j] = neg ? (half_t)1.0f : (half_t)-1.0f;
        }
    const int s0 = blk * 32, s = min(s0 + (l & 31), A.npairs - 1);     // (lanes past the end repeat the last pick)
    const size_t xrow = (size_t)(s / A.topk) * A.x_stride;
    const half_t* suh = (const half_t*)((const uint8_t*)A.ptrs[min(max(A.ids[s], 0), A.E - 1)] +
                                        (pj ? A.g.off_suh_u : A.g.off_suh_g));
    for (int kb = ks * kbs; kb < min(nkb, (ks + 1) * kbs); ++kb) {
        half8_t bx[8];                           // xt fragments: k = 16 i + 8 (l / 32) .. + 7
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int k = kb * 128 + i * 16 + (l >> 5) * 8;
            float xv[8];
            ld_x8<DT>(A.x, xrow + k, xv);
            const half8_u sv = *(const half8_u*)(suh + k);
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
                for (int q = 0; q < 4; ++q) {    // rows n = 32 nb + 8 q + 4 (l / 32) + 0..3
                    typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
                    *(half4_t*)(tb + (l & 31) * kXhRow + n2 * 32 + q * 8 + (l >> 5) * 4) =
                        half4_t{to_half(acc[4 * q] * kRsqrt128), to_half(acc[4 * q + 1] * kRsqrt128),
                                to_half(acc[4 * q + 2] * kRsqrt128), to_half(acc[4 * q + 3] * kRsqrt128)};
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {        // the wave's own LDS rows: 8 picks x 128 bytes per store
                const int pr = r * 8 + (l >> 3), col = (l & 7) * 8;
                const half8_t v = *(const half8_t*)(tb + pr * kXhRow + col);
                if (s0 + pr < A.npairs)
                    *(half8_t*)(A.xh + ((size_t)(s0 + pr) * 2 + pj) * H + kb * 128 + hb * 64 + col) = v;
            }
        }
    }
}

__global__ void __launch_bounds__(kPreThreads) grouped_pre_kernel(GroupedArgs A, int ntask, int kbs) {
    __shared__ __align__(16) half_t tbuf[kPreThreads / 64][32 * kXhRow];
    __shared__ uint64_t sw[17];
    if (blockIdx.x == 0) {
        sort_wg(A, (int*)tbuf, sw);
        return;
    }
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int task = (blockIdx.x - 1) * (kPreThreads / 64) + wv;
    if (task >= ntask) return;
    if (A.x_dt == 1) xh_task<1>(A, task, kbs, tbuf[wv]);
    else if (A.x_dt == 2) xh_task<2>(A, task, kbs, tbuf[wv]);
    else xh_task<0>(A, task, kbs, tbuf[wv]);
}

// ---- the two products ----------------------------------------------------------------------------------------------------

// wave-uniform values that the compiler loads per lane, as scalars: a descriptor in vector registers would make every
// buffer load a loop over its lanes
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ const uint8_t* expert_base(const GroupedArgs& A, int e) {
    const uint64_t p = (uint64_t)A.ptrs[e];
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
__device__ __forceinline__ void gateup_item(const GroupedArgs& A, int e, int s0, int rows, int nb, float* ep) {
    constexpr int NB = 1;
    const int I = A.g.I, H = A.g.H, tiles_n = 2 * I / 16, l = lane_id();
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wc = wv & 3, ks = wv >> 2, pj = wc >> 1;
    using B = RegB<K, false, 2>;
    const uint8_t* base = expert_base(A, e);
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
            const half8_u hg = *(const half8_u*)((const half_t*)(base + A.g.off_svh_g) + cb8);
            const half8_u hu = *(const half8_u*)((const half_t*)(base + A.g.off_svh_u) + cb8);
            const half8_u hd = *(const half8_u*)((const half_t*)(base + A.g.off_suh_d) + cb8);
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
__device__ __forceinline__ void gateup_rows(const GroupedArgs& A, int e, int s0, int rows, int nb, uint8_t* lds) {
    const int I = A.g.I, H = A.g.H, tiles_n = 2 * I / 16, l = lane_id();
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int pj = wv / (WV / 2), wc = wv % (WV / 2);
    using B = RegB<K, false, 2>;
    using U = AUnits<NB, WV, 2>;
    const uint8_t* base = expert_base(A, e);
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
    regb_lds_core<K, NB, WV, 2, false, 2>(rw, B::lane_off(tiles_n, pj * (I / 16) + nb * 2 * WV + wc * 4), tiles_n, ra,
                                          soff, H / 64, pj, lds, acc);
    // 16 rows per round through one of two tiles [16][gate 32 WV | up 32 WV]: 16 lanes per (row, 128 columns)
    const int un = threadIdx.x >> 4, rr = un & 15, cb = (un >> 4) * 128 + (l & 15) * 8, ci = nb * 32 * WV + cb;
    const half8_u hg = *(const half8_u*)((const half_t*)(base + A.g.off_svh_g) + ci);
    const half8_u hu = *(const half8_u*)((const half_t*)(base + A.g.off_svh_u) + ci);
    const half8_u hd = *(const half8_u*)((const half_t*)(base + A.g.off_suh_d) + ci);
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
__device__ __forceinline__ void down_rows(const GroupedArgs& A, int e, int s0, int rows, int nt, uint8_t* lds) {
    const int I = A.g.I, H = A.g.H, tiles_n = H / 16, l = lane_id();
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    using B = RegB<K, false, 2>;
    using U = AUnits<NB, WV, 1>;
    const uint8_t* base = expert_base(A, e);
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
        regb_lds_core<K, NB, WV, 1, false, 2>(rw, woff, tiles_n, ra, soff, I / 64, 0, lds, acc);
    } else {
        uint32_t aoff[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int m = 16 * b + (l & 15);
            aoff[b] = m < rows ? (uint32_t)A.perm[s0 + m] * 2u * I + B::a_lane_off() : kOob;
        }
        regb_core<K, NB, false, 2>(rw, woff, tiles_n, ra, aoff, 0, I / 64, acc);
    }
    // 16 rows per round, 16 lanes per (row, 128 columns), two units per thread
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        float* ep = (float*)lds + (b & 1) * 16 * kEpRowW<WV>;
        stash<K, kEpRowW<WV>>(acc[b], ep, wv);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int un = (threadIdx.x >> 4) + i * 4 * WV, rr = un & 15, cb = (un >> 4) * 128 + (l & 15) * 8;
            const int row = 16 * b + rr, ch = nt * 64 * WV + cb;
            const half8_u hs = *(const half8_u*)((const half_t*)(base + A.g.off_svh_d) + ch);
            const int pk = A.perm[s0 + min(row, rows - 1)];
            const float pw = A.w[pk];
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = ep[rr * kEpRowW<WV> + cb + j];
            row_fwht128_signed(v);
            if (row < rows) st_y<TY>(A.y, (size_t)pk * H + ch, v, row_sign() * kRsqrt128 * pw, hs);
        }
    }
}

// One launch per product (two launches, one per item size, left the chip idle behind the longest item of each: a batch
// of 64 rows took 193 us in two, 132 us in one). !BIG (items of up to 4 blocks): 4 waves per SIMD; the items of several blocks come first, then
// those of one. BIG (items of up to 12 blocks): 2 waves per SIMD, block counts below 9 rounded up to 4, 6 or 8.
template <int K, int WV, bool BIG>
__global__ void __launch_bounds__(64 * WV) __attribute__((amdgpu_waves_per_eu(BIG ? 2 : 4)))
grouped_gateup_kernel(GroupedArgs A) {
    constexpr int kLds = std::max(2 * AUnits<BIG ? 12 : 4, WV, 2>::kBuf, 2 * 16 * kEpRowW<WV> * 4);
    __shared__ __align__(16) uint8_t lds[kLds];
    const int nblk = A.g.I / (32 * WV), nmany = uni(A.n_items[BIG ? 0 : 1]);
    int blk = blockIdx.x, a, nb;
    const int bmany = (nmany + 7) / 8 * 8 * nblk;
    if (BIG || blk < bmany) {
        gr_block(blk, nblk, a, nb);
        if (a >= nmany) return;
    } else {
        if constexpr (!BIG) {
            gr_block(blk - bmany, A.g.I / 128, a, nb);
            a += nmany;
            if (a >= A.n_items[0]) return;
            gateup_item<K, WV / 4>(A, uni(A.it_expert[a]), uni(A.it_start[a]), uni(A.it_cnt[a]), nb, (float*)lds);
        }
        return;
    }
    const int e = uni(A.it_expert[a]), s0 = uni(A.it_start[a]), rows = uni(A.it_cnt[a]), bl = (rows + 15) >> 4;
    if constexpr (!BIG) {
        if (bl <= 2) gateup_rows<K, 2, WV>(A, e, s0, rows, nb, lds);
        else if (bl == 3) gateup_rows<K, 3, WV>(A, e, s0, rows, nb, lds);
        else gateup_rows<K, 4, WV>(A, e, s0, rows, nb, lds);
    } else {
        if (bl <= 4) gateup_rows<K, 4, WV>(A, e, s0, rows, nb, lds);
        else if (bl <= 6) gateup_rows<K, 6, WV>(A, e, s0, rows, nb, lds);
        else if (bl <= 8) gateup_rows<K, 8, WV>(A, e, s0, rows, nb, lds);
        else if (bl == 9) gateup_rows<K, 9, WV>(A, e, s0, rows, nb, lds);
        else if (bl == 10) gateup_rows<K, 10, WV>(A, e, s0, rows, nb, lds);
        else if (bl == 11) gateup_rows<K, 11, WV>(A, e, s0, rows, nb, lds);
        else gateup_rows<K, 12, WV>(A, e, s0, rows, nb, lds);
    }
}

template <int K, int WV, bool BIG, typename TY>
__global__ void __launch_bounds__(64 * WV) __attribute__((amdgpu_waves_per_eu(BIG ? 2 : 4)))
grouped_down_kernel(GroupedArgs A) {
    constexpr int kLds = std::max(2 * AUnits<BIG ? 12 : 4, WV, 1>::kBuf, 2 * 16 * kEpRowW<WV> * 4);
    __shared__ __align__(16) uint8_t lds[kLds];
    int a, nt;
    gr_block(blockIdx.x, A.g.H / (64 * WV), a, nt);
    if (a >= A.n_items[0]) return;
    const int e = uni(A.it_expert[a]), s0 = uni(A.it_start[a]), rows = uni(A.it_cnt[a]), bl = (rows + 15) >> 4;
    if constexpr (!BIG) {
        if (bl == 1) down_rows<K, 1, WV, false, TY>(A, e, s0, rows, nt, lds);
        else if (bl == 2) down_rows<K, 2, WV, true, TY>(A, e, s0, rows, nt, lds);
        else if (bl == 3) down_rows<K, 3, WV, true, TY>(A, e, s0, rows, nt, lds);
        else down_rows<K, 4, WV, true, TY>(A, e, s0, rows, nt, lds);
    } else {
        if (bl <= 4) down_rows<K, 4, WV, true, TY>(A, e, s0, rows, nt, lds);
        else if (bl <= 6) down_rows<K, 6, WV, true, TY>(A, e, s0, rows, nt, lds);
        else if (bl <= 8) down_rows<K, 8, WV, true, TY>(A, e, s0, rows, nt, lds);
        else if (bl == 9) down_rows<K, 9, WV, true, TY>(A, e, s0, rows, nt, lds);
        else if (bl == 10) down_rows<K, 10, WV, true, TY>(A, e, s0, rows, nt, lds);
        else if (bl == 11) down_rows<K, 11, WV, true, TY>(A, e, s0, rows, nt, lds);
        else down_rows<K, 12, WV, true, TY>(A, e, s0, rows, nt, lds);
    }
}

// out[m][h] = sum over the row's picks, in pick order, of y[m topk + k][h]; one thread per 8 columns. The picks' rows are
// loaded kComb at a time before they are summed (picks past topk repeat the last one and are not summed).
constexpr int kComb = 10;
template <typename TY>
__global__ void __launch_bounds__(128) grouped_combine_kernel(GroupedArgs A) {
    const int H = A.g.H, topk = A.topk, m = blockIdx.x;
    const int h0 = (blockIdx.y * 128 + threadIdx.x) * 8;
    if (h0 >= H) return;
    float acc[8] = {};
    for (int k0 = 0; k0 < topk; k0 += kComb) {
        float v[kComb][8];
#pragma unroll
        for (int k = 0; k < kComb; ++k) {
            const size_t o = ((size_t)m * topk + min(k0 + k, topk - 1)) * H + h0;
            if constexpr (sizeof(TY) == 4) {
                const float4_t a = *(const float4_t*)((const float*)A.y + o), b = *(const float4_t*)((const float*)A.y + o + 4);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    v[k][j] = a[j];
                    v[k][4 + j] = b[j];
                }
            } else {
                const half8_t a = *(const half8_t*)((const half_t*)A.y + o);
#pragma unroll
                for (int j = 0; j < 8; ++j) v[k][j] = (float)a[j];
            }
        }
#pragma unroll
        for (int k = 0; k < kComb; ++k)
            if (k0 + k < topk)
#pragma unroll
                for (int j = 0; j < 8; ++j) acc[j] += v[k][j];
    }
    const size_t oo = (size_t)m * A.out_stride + h0;
    // one 16-byte store per 8 outputs when the row start allows it (16-bit outputs, 8-aligned offsets)
    if (A.x_dt != 2 && (A.out_stride & 7) == 0 && ((uintptr_t)A.out & 15) == 0) {
        uint32_t w[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            w[j] = A.x_dt == 1 ? (uint32_t)f32_to_bf16(acc[2 * j]) | ((uint32_t)f32_to_bf16(acc[2 * j + 1]) << 16)
                               : (uint32_t)__builtin_bit_cast(uint16_t, (half_t)acc[2 * j]) |
                                     ((uint32_t)__builtin_bit_cast(uint16_t, (half_t)acc[2 * j + 1]) << 16);
        *(uint4*)((uint16_t*)A.out + oo) = make_uint4(w[0], w[1], w[2], w[3]);
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) st_act(A.out, A.x_dt, oo + j, acc[j]);
    }
}

// ---- host --------------------------------------------------------------------------------------------------------------

// an upper bound of a call's items: every expert's last one, and one more per 64 picks (items are cut at 64 rows or more)
static size_t max_items(size_t np, int E) { return std::min<size_t>(np, (size_t)E) + np / 64; }

// rows of one pass: byte offsets into xh and y stay below 2 GiB (kOob), item counts below 16 bits
static int pass_rows(int M, int topk, int H, int I) {
    const int64_t np = std::min<int64_t>(((int64_t)1 << 31) / (4 * (int64_t)std::max(H, I)) - 1, 1 << 20);
    return (int)std::max<int64_t>(1, std::min<int64_t>(M, np / topk));
}

size_t grouped_workspace_bytes(int M, int topk, int H, int I, int E, bool y32) {
    const size_t np = (size_t)pass_rows(M, topk, H, I) * topk;
    return align256((3 * max_items(np, E) + 2) * 4) + align256(np * 4) + align256(np * 4 * H) + align256(np * 2 * I) +
           align256(np * H * (y32 ? 4 : 2));
}

template <int K>
static void launch_products(const GroupedArgs& a, bool y32, hipStream_t s) {
    const size_t np = a.npairs, mi = max_items(np, a.E);
    auto g8 = [](size_t items) { return (unsigned)((items + 7) / 8 * 8); };
    const int I = a.g.I, H = a.g.H;
    const bool big = a.rmax > 64;
    auto run = [&](auto kern, unsigned grid, int nt) { hipLaunchKernelGGL(kern, dim3(grid), dim3(nt), 0, s, a); };
    // items of several blocks hold at least 17 rows each
    const unsigned many = g8(np / 17);
    if (I % 256 == 0) {
        if (big) run(grouped_gateup_kernel<K, 8, true>, g8(mi) * (I / 256), 512);
        else run(grouped_gateup_kernel<K, 8, false>, many * (I / 256) + g8(std::min<size_t>(np, a.E)) * (I / 128), 512);
    } else {
        if (big) run(grouped_gateup_kernel<K, 4, true>, g8(mi) * (I / 128), 256);
        else run(grouped_gateup_kernel<K, 4, false>, (many + g8(std::min<size_t>(np, a.E))) * (I / 128), 256);
    }
    auto down = [&](auto ty) {
        using TY = decltype(ty);
        if (H % 512 == 0) {
            if (big) run(grouped_down_kernel<K, 8, true, TY>, g8(mi) * (H / 512), 512);
            else run(grouped_down_kernel<K, 8, false, TY>, g8(mi) * (H / 512), 512);
        } else {
            if (big) run(grouped_down_kernel<K, 4, true, TY>, g8(mi) * (H / 256), 256);
            else run(grouped_down_kernel<K, 4, false, TY>, g8(mi) * (H / 256), 256);
        }
    };
    if (y32) down(float{});
    else down(half_t{});
}

static hipError_t launch_pass(GroupedArgs a, bool y32, void* ws, hipStream_t s) {
    const size_t np = (size_t)a.npairs, mi = max_items(np, a.E);
    // Items of up to 64 rows run 4 waves per SIMD; of up to 192 rows 2 (the accumulators), but decode once where the
    // others decode three times. With 56 rows per expert on average and more, 64-row items would cut most experts
    // (H 4096 / I 1536 / K 2, 777 tokens of 49 rows per expert: 64-row items 533 us, items of up to 128 rows 603 us).
    a.rmax = np > (size_t)56 * a.E ? 192 : 64;
    uint8_t* p = (uint8_t*)ws;
    auto take = [&p](size_t n) { uint8_t* q = p; p += align256(n); return q; };
    int* it = (int*)take((3 * mi + 2) * 4);
    a.it_expert = it;
    a.it_start = it + mi;
    a.it_cnt = it + 2 * mi;
    a.n_items = it + 3 * mi;
    a.perm = (int*)take(np * 4);
    a.xh = (half_t*)take(np * 4 * a.g.H);
    a.abuf = (half_t*)take(np * 2 * a.g.I);
    a.y = take(np * a.g.H * (y32 ? 4 : 2));
    const int nkb = a.g.H / 128, nblk = (a.npairs + 31) / 32;
    int kbs = 1;                                 // 128-blocks per wave
    while (kbs < nkb && 2 * nblk * ((nkb + kbs - 1) / kbs) > 65536) kbs *= 2;
    const int ntask = 2 * nblk * ((nkb + kbs - 1) / kbs);
    hipLaunchKernelGGL(grouped_pre_kernel, dim3(1 + (unsigned)((ntask + 15) / 16)), dim3(kPreThreads), 0, s, a, ntask, kbs);
    switch (a.g.K) {
        case 2: launch_products<2>(a, y32, s); break;
        case 3: launch_products<3>(a, y32, s); break;
        case 4: launch_products<4>(a, y32, s); break;
        default: return hipErrorInvalidValue;
    }
    const dim3 gc((unsigned)a.M, (unsigned)((a.g.H + 1023) / 1024));
    if (y32) hipLaunchKernelGGL(grouped_combine_kernel<float>, gc, dim3(128), 0, s, a);
    else hipLaunchKernelGGL(grouped_combine_kernel<half_t>, gc, dim3(128), 0, s, a);
    return hipGetLastError();
}

// calls beyond one pass's limits run their rows in passes of the same workspace (a row depends on no other row)
hipError_t launch_grouped(const GroupedArgs& a0, bool y32, void* ws, hipStream_t s) {
    const int step = pass_rows(a0.M, a0.topk, a0.g.H, a0.g.I), esz = a0.x_dt == 2 ? 4 : 2;
    for (int m0 = 0; m0 < a0.M; m0 += step) {
        GroupedArgs a = a0;
        a.M = std::min(step, a0.M - m0);
        a.npairs = a.M * a.topk;
        a.x = (const uint8_t*)a0.x + (int64_t)m0 * a0.x_stride * esz;
        a.out = (uint8_t*)a0.out + (int64_t)m0 * a0.out_stride * esz;
        a.ids = a0.ids + (size_t)m0 * a.topk;
        a.w = a0.w + (size_t)m0 * a.topk;
        const hipError_t e = launch_pass(a, y32, ws, s);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace exl3
