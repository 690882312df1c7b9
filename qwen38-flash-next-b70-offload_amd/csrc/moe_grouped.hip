// Routed experts with the picks grouped by expert (decode batches and prompts): every expert's trellis is decoded once
// per item of up to 64 or 192 rows, straight into MFMA B registers (exl3_regb.cuh).
//
//   scales   above 16 picks per expert: the input scales of the experts in use, once each, into the workspace
//   pre      one launch: workgroup 0 sorts the picks by expert and cuts them into items (longest first), the others
//            write the input Hadamards xh of every (pick, projection), which need no sort
//   gate/up  per (item, 32 WV columns of I), WV waves of 64 columns, half of them on each projection; the rows gathered
//            by pick; epilogue through LDS: g/u Hadamards, SwiGLU, * suh_d, Hadamard -> abuf[pick] (fp16)
//   down     per (item, 64 WV columns of H), K = I, the same core; output Hadamard * (w * svh_d) -> y[pick]
//   combine  out[m] = sum over the row's picks of y, in pick order (fp32)
// A cached call's misses are copied into their slots by workgroups of the same launches (FILL, exl3_fill.cuh).
// (reference: kernels/moe-a8/exl3_moe.a8.sycl:121-395, 422-635, 639-680, with the same fp16 rounding points.)
//
// What bounds them: the decode's VALU work, 3.5 instructions per weight (bfe, mul_lo, sad, half a pk_fma) at 4.2 to 4.6
// clocks each per wave of 64. At H 2048 / I 512 / K 3 with all 512 experts active that is 155 us per layer at 2.4 GHz
// against 97 us for the 612 MB of weights at 6.3 TB/s; with up to 16 rows per expert (301 tokens, top-10) gate/up
// takes 150-170 us and down 85-98 us, 89 % and 79 % of their VALU cycles issuing. Columns are split over waves, not K,
// so that a weight is decoded by one wave and multiplied into every row, and nothing is exchanged before the epilogue.
// Whole layers, bf16, before (one decode per pick, or a core that decodes into LDS for 192-row passes) and now:
// 16 Zipf rows 104 -> 63 us, 64 rows 399 -> 120 us, 301 tokens 605 -> 232 us, 2,048 tokens 726 -> 363 us, 8,192 tokens
// 1,269 -> 1,072 us; H 4096 / I 1536, 128 experts, top-8, K 2, 777 tokens: 861 -> 465 us.
#include "exl3_common.cuh"
#include "exl3_fill.cuh"
#include "exl3_geom.h"
#include "exl3_kernels.h"
#include "exl3_regb.cuh"
#include "exl3_xh.cuh"

#include <algorithm>

namespace exl3 {

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
// that the longest start first. n_items[0]: all items, [1]: those of more than one block. With big_n, the experts outside
// [hbm_lo, hbm_hi) of more than 64 rows are cut at 192 rows (5 blocks and more) into a list of their own.
__device__ __forceinline__ void emit_items(const GroupedArgs& A, int e, int st, int tot, uint64_t* sw) {
    int64_t blob = 0;
    if (tot) {                                   // (a miss of a cached call: its new slot)
        blob = A.ptrs[e];
        if (A.f.list && A.f.fill[e]) blob = A.f.fill[e];
    }
    const int rmax = A.big_n && tot > 64 && (blob < A.hbm_lo || blob >= A.hbm_hi) ? 192 : A.rmax;
    const int n = (tot + rmax - 1) / rmax, nb = n ? ((tot + n - 1) / n + 15) >> 4 : 0;       // items, blocks of each
    int above = 0;
    for (int g = A.big_n ? 2 : (A.rmax + 63) / 64 - 1; g >= 0; --g) {      // block counts 4 g + 1 .. 4 g + 4
        const bool big = A.big_n && g > 0;
        if (A.big_n && g == 0) {
            if (threadIdx.x == 0) A.big_n[0] = above;
            above = 0;
        }
        uint64_t tt;
        const uint64_t ex = block_scan64(nb > 4 * g && nb <= 4 * g + 4 ? (uint64_t)n << (16 * (nb - 1 - 4 * g)) : 0ull, sw, tt);
#pragma unroll
        for (int k = 4; k >= 1; --k) {
            if (4 * g + k == nb) {
                int p = above + (int)((ex >> (16 * (k - 1))) & 0xFFFF);
                for (int i = 0; i < n; ++i, ++p) {
                    (big ? A.big_blob : A.it_blob)[p] = blob;
                    (big ? A.big_start : A.it_start)[p] = st + i * 16 * nb;
                    (big ? A.big_cnt : A.it_cnt)[p] = min(16 * nb, tot - i * 16 * nb);
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

// ---- input scales ------------------------------------------------------------------------------------------------------
// The input Hadamards run in pick order and read an expert's input scales for each of its picks: 8 KB per pick and expert
// of H 2048. That is cache traffic for an expert in HBM, but host memory is not cached, so with a third of 512 experts
// read over PCIe and 160 picks per expert it was 230 MB next to the 412 MB of their records (8,192 tokens 12.7 ms per
// layer, 8.2 ms with the copies and with down's output scales loaded once; with every expert in HBM 1.09 ms either way).
// So each expert's scales are copied once: a workgroup per kScaleExperts experts looks for them in the ids (an expert
// without picks may have no blob) and copies those that it finds.
constexpr int kScaleExperts = 4;
__global__ void __launch_bounds__(1024) grouped_scales_kernel(GroupedArgs A) {
    __shared__ int used[kScaleExperts];
    const int e0 = blockIdx.x * kScaleExperts, t = threadIdx.x;
    if (t < kScaleExperts) used[t] = 0;
    __syncthreads();
    for (int i0 = t; i0 < A.npairs; i0 += 8 * 1024) {
        int e[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) e[j] = min(max(A.ids[min(i0 + j * 1024, A.npairs - 1)], 0), A.E - 1) - e0;
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if ((unsigned)e[j] < (unsigned)kScaleExperts) used[e[j]] = 1;
    }
    __syncthreads();
    // 8 values per thread; suh_u follows suh_g
    const int n = 2 * A.g.H;
    for (int i = t * 8; i < kScaleExperts * n; i += 8 * 1024) {
        const int e = i / n, c = i % n;
        if (used[e]) *(half8_t*)(A.suh + (size_t)e0 * n + i) = ld_half8((const uint8_t*)A.ptrs[e0 + e] + A.g.off_suh_g + 2 * c);
    }
}

// ---- input Hadamards ---------------------------------------------------------------------------------------------------
// xh[pick][pj][kb * 128 ..] = fp16(H(fp16(x[row] suh_pj)) / sqrt 128), one wave per (4 picks, kbs 128-blocks) and both
// projections: 16 lanes hold a pick's block, 8 values each (row_fwht128_signed). Few registers, no LDS, full cache lines
// in and out. As MFMA products with H128 (32 picks per wave, through LDS twice, 128 VGPRs) the blocks of a wave ran one
// after the other, 6 us each: 250-280 us at 8,192 tokens, 82 us at 2,048; so 201 and 57 us, with 671 MB written (107 us at
// 6.3 TB/s) at 8,192.
template <int DT>
__device__ __forceinline__ void xh_task(const GroupedArgs& A, int task, int kbs) {
    const int H = A.g.H, nkb = H / 128, nks = (nkb + kbs - 1) / kbs, l = lane_id();
    const int ks = task % nks, p = task / nks * 4 + (l >> 4), c = (l & 15) * 8;
    const int s = min(p, A.npairs - 1);          // (lanes past the end repeat the last pick and store nothing)
    const size_t xo = (size_t)(s / A.topk) * A.x_stride + c;
    const int e = min(max(A.ids[s], 0), A.E - 1);
    const uint8_t* su = A.suh ? (const uint8_t*)(A.suh + (size_t)e * 2 * H + c)
                              : (const uint8_t*)A.ptrs[e] + A.g.off_suh_g + 2 * c;
    half_t* o = A.xh + (size_t)s * 2 * H + c;
    const float rs = row_sign() * kRsqrt128;
    const int kb1 = min(nkb, (ks + 1) * kbs);
    XRaw<DT> x;
    half8_u sg, sv;
    auto load = [&](int kb) {
        ld_x8<DT>(A.x, xo + kb * 128, x);
        sg = ld_half8(su + kb * 256);
        sv = ld_half8(su + 2 * H + kb * 256);    // suh_u follows suh_g
    };
    load(ks * kbs);
    for (int kb = ks * kbs; kb < kb1; ++kb) {
        float g[8], u[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            g[j] = x_su<DT>(x, j, sg[j]);
            u[j] = x_su<DT>(x, j, sv[j]);
        }
        load(min(kb + 1, nkb - 1));              // the next block's, while this one is transformed
        row_fwht128_signed(g);
        row_fwht128_signed(u);
        half8_t og, ou;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            og[j] = to_half(g[j] * rs);
            ou[j] = to_half(u[j] * rs);
        }
        if (p < A.npairs) {
            *(half8_t*)(o + kb * 128) = og;
            *(half8_t*)(o + H + kb * 128) = ou;
        }
    }
}

template <bool FILL>
__global__ void __launch_bounds__(kPreThreads) __attribute__((amdgpu_waves_per_eu(8)))
grouped_pre_kernel(GroupedArgs A, int ntask, int kbs) {
    __shared__ int off[kMaxExperts];
    __shared__ uint64_t sw[17];
    if (blockIdx.x == 0) {
        sort_wg(A, off, sw);
        return;
    }
    int blk = blockIdx.x - 1;
    if constexpr (FILL) {                        // a cached call's misses: what gate/up reads of them
        if (blk < fill_workgroups(kPreThreads)) {
            fill_part<kPreThreads>(A, 0, blk);
            if (A.rmax > 64) fill_part<kPreThreads>(A, 1, blk);   // (the large gate/up kernel copies nothing)
            return;
        }
        blk -= fill_workgroups(kPreThreads);
    }
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int task = blk * (kPreThreads / 64) + wv;
    if (task >= ntask) return;                   // (whole waves: the transforms need every lane)
    if (A.x_dt == 1) xh_task<1>(A, task, kbs);
    else if (A.x_dt == 2) xh_task<2>(A, task, kbs);
    else xh_task<0>(A, task, kbs);
}

// out[m][h] = sum over the row's picks, in pick order, of y[m topk + k][h]; one thread per 8 columns. The picks' rows are
// loaded kComb at a time before they are summed (picks past topk repeat the last one and are not summed).
constexpr int kComb = 10;
template <typename TY, bool FILL>
__global__ void __launch_bounds__(128) grouped_combine_kernel(GroupedArgs A) {
    const int H = A.g.H, topk = A.topk, m = blockIdx.x;
    const int h0 = (blockIdx.y * 128 + threadIdx.x) * 8;
    if (FILL && blockIdx.x == 0 && blockIdx.y == 0)              // a cached call's misses are in their slots: commit them
        for (int mi = threadIdx.x; mi < A.f.list[0]; mi += 128) {
            const int e = A.f.list[1 + mi];
            A.f.ptrs[e] = A.f.fill[e];
            A.f.fill[e] = 0;
        }
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

// rows of one pass: byte offsets into xh and y stay below 2 GiB (kOob), item counts below 16 bits
static int pass_rows(int M, int topk, int H, int I) {
    const int64_t np = std::min<int64_t>(((int64_t)1 << 31) / (4 * (int64_t)std::max(H, I)) - 1, 1 << 20);
    return (int)std::max<int64_t>(1, std::min<int64_t>(M, np / topk));
}

// The scales are copied from 2 picks per expert on where experts may be in host memory (300 tokens, a third of the experts
// there: 3,805 us without, 3,755 with the copies), else from 16 on, for a table of unknown make (301 tokens in HBM: 235
// without, 240 us with them). The workspace has room for min(E, np / 2) experts' scales (np / 16 at the decode sizes, which
// copy from 16 on), which grows with both
static bool grouped_scales(size_t np, int E, bool host) { return np > (size_t)(host ? 2 : 16) * E; }
// the lists of an upper bound of n items and their counts
static size_t list_bytes(size_t n) { return align256((4 * n + 2) * 4); }
static size_t big_items(size_t np) { return np / 65; }           // (an expert of more than 64 rows has 65 or more per item)

// y starts 1 KiB into a page of 4 KiB: the combine reads the picks' rows and writes the output's at once, and with both on
// page boundaries their lines fall on the same channels (8,192 tokens, H 2048: starts 0 / 256 / 512 / 1,024 / 2,048 / 3,072
// bytes into a page 77 / 72 / 67 / 63 / 75 / 63 us)
constexpr size_t kYPage = 4096;
static uint8_t* y_start(uint8_t* p) { return p + ((1024 - (uintptr_t)p) & (kYPage - 1)); }

size_t grouped_workspace_bytes(int M, int topk, int H, int I, int E, bool y32) {
    const size_t np = (size_t)pass_rows(M, topk, H, I) * topk;
    return list_bytes(grouped_max_items(np, E)) + (y32 ? 0 : list_bytes(big_items(np))) + align256(np * 4) +
           align256(np * 4 * H) + align256(np * 2 * I) + align256(np * H * (y32 ? 4 : 2) + kYPage) +
           align256(std::min<size_t>(E, np / (y32 ? 16 : 2)) * 4 * H);
}

static hipError_t launch_pass(GroupedArgs a, bool y32, void* ws, hipStream_t s) {
    const size_t np = (size_t)a.npairs, mi = grouped_max_items(np, a.E);
    // Items of up to 64 rows run 4 waves per SIMD; of up to 192 rows 2 (the accumulators), but decode once where the
    // others decode three times. With 56 rows per expert on average and more, 64-row items would cut most experts
    // (H 4096 / I 1536 / K 2, 777 tokens of 49 rows per expert: 64-row items 533 us, items of up to 128 rows 603 us).
    const bool host = a.hbm_hi != 0 && !y32, large = a.g.I % 256 == 0 && a.g.H % 512 == 0 && !y32;
    a.rmax = large && np > (size_t)56 * a.E ? 192 : 64;
    uint8_t* p = (uint8_t*)ws;
    auto take = [&p](size_t n) { uint8_t* q = p; p += align256(n); return q; };
    int* it = (int*)take(list_bytes(mi));
    a.it_blob = (int64_t*)it;
    a.it_start = it + 2 * mi;
    a.it_cnt = it + 3 * mi;
    a.n_items = it + 4 * mi;
    // Experts in host memory: each 64-row item would read its expert over PCIe again, so those of more rows run as items of
    // up to 192 rows in launches of their own; only those, since the reads of the others would wait for the HBM experts'
    // items among them. H 2048 / I 512 / K 3, Zipf tokens, a third of the experts in host memory, us without and with: 700
    // tokens 4,104 and 3,780, 1,500 4,592 and 4,013, 2,600 4,857 and 4,190; H 4096 / I 1536 / K 4, 777 tokens 9,835 and 7,750.
    // With every expert in HBM the added launches and the copied scales cost 3-10 us (301 tokens 235 and 243).
    if (host && large && a.rmax == 64) {
        const size_t mb = big_items(np);
        int* b = (int*)take(list_bytes(mb));
        a.big_blob = (int64_t*)b;
        a.big_start = b + 2 * mb;
        a.big_cnt = b + 3 * mb;
        a.big_n = b + 4 * mb;
    }
    a.perm = (int*)take(np * 4);
    a.xh = (half_t*)take(np * 4 * a.g.H);
    a.abuf = (half_t*)take(np * 2 * a.g.I);
    a.y = y_start(take(np * a.g.H * (y32 ? 4 : 2) + kYPage));
    a.suh = nullptr;
    if (grouped_scales(np, a.E, host)) {
        a.suh = (half_t*)take((size_t)a.E * 4 * a.g.H);
        hipLaunchKernelGGL(grouped_scales_kernel, dim3((unsigned)((a.E + kScaleExperts - 1) / kScaleExperts)), dim3(1024), 0, s, a);
    }
    const int nkb = a.g.H / 128, nq = (a.npairs + 3) / 4;
    // 128-blocks per wave: one while the waves do not fill the chip several times over, then up to 4, which hides a
    // wave's own table lookups (8,192 tokens: 1 / 2 / 4 / 8 blocks 230 / 207 / 201 / 207 us; 16 rows: 5.4 / 5.6 / 8.6 us)
    int kbs = 1;
    while (kbs < 4 && nq * ((nkb + kbs - 1) / kbs) > 32768) kbs *= 2;
    const int ntask = nq * ((nkb + kbs - 1) / kbs);
    const unsigned grid = 1 + (unsigned)((ntask + 15) / 16);
    auto pre = [&](auto kern, unsigned n) { hipLaunchKernelGGL(kern, dim3(n), dim3(kPreThreads), 0, s, a, ntask, kbs); };
    if (a.f.list) pre(grouped_pre_kernel<true>, fill_workgroups(kPreThreads) + grid);
    else pre(grouped_pre_kernel<false>, grid);
    switch (a.g.K) {
        case 2: launch_products<2>(a, y32, s); break;
        case 3: launch_products<3>(a, y32, s); break;
        case 4: launch_products<4>(a, y32, s); break;
        default: return hipErrorInvalidValue;
    }
    const dim3 gc((unsigned)a.M, (unsigned)((a.g.H + 1023) / 1024));
    auto combine = [&](auto kern) { hipLaunchKernelGGL(kern, gc, dim3(128), 0, s, a); };
    if (a.f.list) combine(y32 ? grouped_combine_kernel<float, true> : grouped_combine_kernel<half_t, true>);
    else combine(y32 ? grouped_combine_kernel<float, false> : grouped_combine_kernel<half_t, false>);
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
        if (m0) a.f = FillArgs{};                // (committed by the first pass)
        const hipError_t e = launch_pass(a, y32, ws, s);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace exl3
