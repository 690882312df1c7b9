// The token sort as its own call (exl3_moe_align; reference: launch_align, kernels/moe-a8/exl3_moe.a8.sycl:639-680):
// three small kernels (count per chunk of 1,024 pairs, scan, scatter), pairs sorted by expert in ascending pair order
// inside an expert (deterministic; wave ballots for in-chunk ranks).
#include "exl3_common.cuh"
#include "exl3_kernels.h"

namespace exl3 {

constexpr int kAlignChunk = 1024;

// ---- block scan helpers (1,024 threads) ---------------------------------------------------------------------------
__device__ __forceinline__ int wave_incl_scan(int v) {
    const int l = lane_id();
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int t = __shfl_up(v, d, 64);
        if (l >= d) v += t;
    }
    return v;
}
// exclusive scan over the block; tot = block sum. sw: LDS [16 + 1]
__device__ __forceinline__ int block_scan_1024(int v, int* sw, int& tot) {
    const int l = lane_id(), w = threadIdx.x >> 6;
    const int inc = wave_incl_scan(v);
    if (l == 63) sw[w] = inc;
    __syncthreads();
    if (w == 0) {
        const int x = l < 16 ? sw[l] : 0;
        const int xi = wave_incl_scan(x);
        if (l < 16) sw[l] = xi - x;
        if (l == 15) sw[16] = xi;
    }
    __syncthreads();
    const int r = sw[w] + inc - v;
    tot = sw[16];
    __syncthreads();
    return r;
}

// ---- align -----------------------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(1024) align_count_kernel(const int32_t* ids, int npairs, int E, int* chunk_cnt) {
    extern __shared__ int hist[];                 // [E]
    for (int e = threadIdx.x; e < E; e += 1024) hist[e] = 0;
    __syncthreads();
    const int i = blockIdx.x * kAlignChunk + threadIdx.x;
    if (i < npairs) atomicAdd(&hist[min(max(ids[i], 0), E - 1)], 1);
    __syncthreads();
    for (int e = threadIdx.x; e < E; e += 1024) chunk_cnt[(size_t)blockIdx.x * E + e] = hist[e];
}

// per expert (one thread each, E <= 1024): totals, starts, active list, padded starts; chunk counts -> chunk offsets
__global__ void __launch_bounds__(1024) align_scan_kernel(int nchunks, int E, int pad, int* chunk_cnt, AlignOut o) {
    __shared__ int sw[17];
    const int e = threadIdx.x;
    constexpr int kB = 16;                        // chunk counts loaded together (clamped indices: no branch per load)
    int tot = 0;
    if (e < E)
        for (int c0 = 0; c0 < nchunks; c0 += kB) {
            int v[kB];
#pragma unroll
            for (int j = 0; j < kB; ++j) v[j] = chunk_cnt[(size_t)min(c0 + j, nchunks - 1) * E + e];
#pragma unroll
            for (int j = 0; j < kB; ++j) tot += c0 + j < nchunks ? v[j] : 0;
        }
    int all;
    const int st = block_scan_1024(e < E ? tot : 0, sw, all);
    const int act = (e < E && tot > 0) ? 1 : 0;
    int nact;
    const int ai = block_scan_1024(act, sw, nact);
    const int pc = (tot + pad - 1) / pad * pad;
    int ptot;
    const int pst = block_scan_1024(e < E ? pc : 0, sw, ptot);
    if (act) {
        o.act_expert[ai] = e;
        o.act_start[ai] = st;
        o.act_cnt[ai] = tot;
        o.act_pstart[ai] = pst;
    }
    if (e == 0) o.n_act[0] = nact;
    if (e < E) {                                  // the counts become each chunk's first position of expert e
        int run = st;
        for (int c0 = 0; c0 < nchunks; c0 += kB) {
            int v[kB];
#pragma unroll
            for (int j = 0; j < kB; ++j) v[j] = chunk_cnt[(size_t)min(c0 + j, nchunks - 1) * E + e];
#pragma unroll
            for (int j = 0; j < kB; ++j)
                if (c0 + j < nchunks) {
                    chunk_cnt[(size_t)(c0 + j) * E + e] = run;
                    run += v[j];
                }
        }
    }
}

// positions: chunk offset of the expert + pairs of that expert in earlier waves of the chunk + rank inside the wave
__global__ void __launch_bounds__(1024) align_scatter_kernel(const int32_t* ids, const float* w, int npairs, int topk,
                                                             int E, const int* chunk_off, AlignOut o) {
    extern __shared__ int wh[];                   // [16][E] per-wave counts, then per-wave offsets
    for (int i = threadIdx.x; i < 16 * E; i += 1024) wh[i] = 0;
    __syncthreads();
    const int l = lane_id(), wv = threadIdx.x >> 6;
    const int i = blockIdx.x * kAlignChunk + threadIdx.x;
    const bool valid = i < npairs;
    const int e = valid ? min(max(ids[i], 0), E - 1) : -1;
    uint64_t todo = __ballot(valid);
    int rank = 0;
    while (todo) {
        const int leader = __builtin_ctzll(todo);
        const int ev = __shfl(e, leader, 64);
        const uint64_t m = __ballot(valid && e == ev);
        if (valid && e == ev) rank = __popcll(m & ((1ull << l) - 1));
        if (l == leader) wh[wv * E + ev] = __popcll(m);
        todo &= ~m;
    }
    __syncthreads();
    for (int x = threadIdx.x; x < E; x += 1024) {
        int run = 0;
        for (int q = 0; q < 16; ++q) {
            const int v = wh[q * E + x];
            wh[q * E + x] = run;
            run += v;
        }
    }
    __syncthreads();
    if (valid) {
        const int pos = chunk_off[(size_t)blockIdx.x * E + e] + wh[wv * E + e] + rank;
        o.pair_tok[pos] = i / topk;
        o.pair_w[pos] = w[i];
        o.pair_of[i] = pos;
    }
}

hipError_t launch_align(const int32_t* ids, const float* w, int npairs, int topk, int E, int pad, int* chunk_scratch,
                        const AlignOut& o, hipStream_t s) {
    const int nch = npairs > 0 ? (npairs + kAlignChunk - 1) / kAlignChunk : 0;
    if (nch == 0) {                               // no pairs: empty lists, n_act = 0 (no memset: graph-safe)
        hipLaunchKernelGGL(align_scan_kernel, dim3(1), dim3(1024), 0, s, 0, E, pad, chunk_scratch, o);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(align_count_kernel, dim3(nch), dim3(1024), E * sizeof(int), s, ids, npairs, E, chunk_scratch);
    hipLaunchKernelGGL(align_scan_kernel, dim3(1), dim3(1024), 0, s, nch, E, pad, chunk_scratch, o);
    hipLaunchKernelGGL(align_scatter_kernel, dim3(nch), dim3(1024), 16 * E * sizeof(int), s, ids, w, npairs, topk, E,
                       (const int*)chunk_scratch, o);
    return hipGetLastError();
}

size_t align_scratch_bytes(int npairs, int E) {
    return (size_t)((npairs + kAlignChunk - 1) / kAlignChunk) * E * 4;
}

}  // namespace exl3
