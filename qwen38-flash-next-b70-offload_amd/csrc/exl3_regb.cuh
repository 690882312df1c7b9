// Trellis weights decoded straight into MFMA B registers (v_mfma_f32_16x16x32_f16) on gfx950, shared by the grouped
// expert kernels and the dense linear: a wave multiplies up to 16 NB activation rows into 64 columns (4 tile-columns)
// over K chunks of 64 rows (4 tile-rows), with no LDS and no barrier between its loads, its decode and its MFMAs.
//
// Lane l = 16 q + n of a 16x16x32 MFMA holds, as B, 8 of the 32 k rows of column n; the rows may be taken in any order
// that the A fragments share. A period holds two columns (c and c + 8 of a tile: h = 0, 1), so lane n decodes tile-
// column n >> 3 of a pair and column n & 7 (+ 8 h), and the k-groups q are chosen so that a lane's 8 rows of a column
// come from its own words:
//   V = 32 (K = 3, 5): one period = all 16 rows. q = tile-row of the chunk (in the order of krow), fragment f = rows
//     8 f .. 8 f + 7 of it.
//   V = 16 (K = 2, 6) and V = 8 (K = 4): f = pair of tile-rows, q >> 1 the tile-row of the pair and b = q & 1 the rows
//     {4 b .. 4 b + 3, 8 + 4 b .. 8 + 4 b + 3}: one period at V = 16, two neighbouring ones at V = 8.
#pragma once
#include <type_traits>

#include "exl3_common.cuh"

namespace exl3 {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// two decoded weights (states s0 and s1, s0 in the low half) as fp16, bit-exact (cb_w2 / cb_w2_lcg)
template <int CB>
__device__ __forceinline__ uint32_t cb_pair(uint32_t s0, uint32_t s1) {
    if constexpr (CB == 2) return __builtin_bit_cast(uint32_t, cb_w2(s0, s1));
    else return __builtin_bit_cast(uint32_t, cb_w2_lcg<CB>(s0, s1));
}

template <int K, bool NAT, int CB>
struct RegB {
    using GM = Geo<K>;
    static constexpr int D = GM::D, V = GM::V, G = GM::G, W = GM::W;
    static constexpr bool F8 = V == 32;
    static constexpr int NP = V == 8 ? 2 : 1;        // periods of a lane per tile
    // PLANAR4 words of K = 3: a load takes whole 128-byte lines, 2 tile-rows x 4 tile-columns, and one permlane16 swap per
    // word of the two loads gives the lanes their tile-column pairs, with the tile-rows in the order 0, 2, 1, 3. Loads
    // of 2 columns of 4 tile-rows take half lines: with a third of the experts in host memory 50.6 GB/s over PCIe
    // against 52.9 with whole lines, 301 tokens 254 against 250 us
    static constexpr bool SWAP = F8 && !NAT;
    static constexpr int SPC = F8 ? 1 : 2;           // steps (tile-row groups) of a chunk
    static constexpr int NW = SPC * 2 * NP * D;      // words of a lane per chunk
    static_assert(V == 32 || V == 16 || V == 8, "periods of 32, 16 or 8 values");

    // byte offset of this lane's first word of chunk 0 in the strip of tile-columns ct0 .. ct0 + 3
    __device__ __forceinline__ static uint32_t lane_off(int tiles_n, int ct0) {
        const int l = lane_id(), q = l >> 4, c = (l >> 3) & (SWAP ? 3 : 1), n = l & 7;
        const int r = SWAP ? l >> 5 : F8 ? q : q >> 1;
        const int p = F8 ? n : (V == 16 ? 2 * n + (q & 1) : 4 * n + 2 * (q & 1));
        return 4u * (uint32_t)(NAT ? word_off_nat<K>(r, tiles_n, ct0 + c, p, 0) : word_off<K>(r, tiles_n, ct0 + c, p, 0));
    }
    // bytes between chunks
    __device__ __forceinline__ static uint32_t chunk_bytes(int tiles_n) { return 16u * (uint32_t)tiles_n * W; }

    // the words of the chunk at byte offset off (lane_off + chunk * chunk_bytes; an offset past the descriptor's range
    // reads zero without touching memory)
    template <typename R>
    __device__ __forceinline__ static void load(uint32_t (&w)[NW], R rsrc, uint32_t off, int tiles_n) {
        constexpr int kTwoTiles = NAT || D == 1 ? 2 * W : 2 * G;           // words from column pair 0 to 1
        constexpr int kPlane = NAT || D == 1 ? 1 : 4 * G;                  // words from word i to i + 1 of a period
        if constexpr (SWAP) {                        // order [tile-row pair][word], see arrange
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int i = 0; i < D; ++i)
                    w[h * D + i] = __builtin_amdgcn_raw_buffer_load_b32(
                        rsrc, (int)(off + h * 8u * (uint32_t)tiles_n * W + 4u * (i * kPlane)), 0, 2);   // 2: nt
            return;
        }
#pragma unroll
        for (int s = 0; s < SPC; ++s) {
            const uint32_t o = off + (s ? 8u * (uint32_t)tiles_n * W : 0u);
#pragma unroll
            for (int cc = 0; cc < 2; ++cc) {
                uint32_t* v = w + (s * 2 + cc) * NP * D;
                if constexpr (NP == 2) {             // the two neighbouring words in one load
                    const auto t = __builtin_amdgcn_raw_buffer_load_b64(rsrc, (int)(o + 4u * cc * kTwoTiles), 0, 2);
                    v[0] = t[0];
                    v[1] = t[1];
                } else {
#pragma unroll
                    for (int i = 0; i < D; ++i)
                        v[i] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)(o + 4u * (cc * kTwoTiles + i * kPlane)), 0, 2);
                }
            }
        }
    }
    // the loaded words into the order [step][column pair][period][word] (before prep, once they are needed)
    __device__ __forceinline__ static void arrange(uint32_t (&w)[NW]) {
        if constexpr (SWAP) {
#pragma unroll
            for (int i = 0; i < D; ++i) {
                const auto t = __builtin_amdgcn_permlane16_swap(w[i], w[D + i], false, false);
                w[i] = t[0];
                w[D + i] = t[1];
            }
        }
    }
    // tile-row of k-group q (V = 32)
    __device__ __forceinline__ static int krow(int q) { return SWAP ? ((q & 1) << 1) | (q >> 1) : q; }

    // the lane holding the period before this lane's first one (the trellis is circular in a tile)
    __device__ __forceinline__ static int prev_lane() {
        const int l = lane_id();
        if constexpr (F8) return (l & ~7) | ((l + 7) & 7);
        return (l & 16) ? l - 16 : (((l + 16) & ~7) | ((l + 7) & 7));
    }

    struct Dec { Period<K> p[NP]; };
    __device__ __forceinline__ static void prep(Dec& d, const uint32_t (&w)[NW], int s, int cc, int src) {
        const uint32_t* v = w + (s * 2 + cc) * NP * D;
        const uint32_t prev = (uint32_t)__shfl((int)v[NP * D - 1], src, 64);
        d.p[0].set(v, prev);
        if constexpr (NP == 2) d.p[1].set(v + D, v[D - 1]);
    }
    // fragment f of column half h (f: only V = 32 keeps both fragments in one period)
    template <int f, int h>
    __device__ __forceinline__ static half8_t frag(const Dec& d) {
        u32x4_t r;
        if constexpr (F8) {
            constexpr int u = 2 * f + 4 * h;
            r = u32x4_t{pr<u>(d.p[0]), pr<u + 8>(d.p[0]), pr<u + 16>(d.p[0]), pr<u + 24>(d.p[0])};
        } else if constexpr (V == 16) {
            constexpr int u = 4 * h;
            r = u32x4_t{pr<u>(d.p[0]), pr<u + 8>(d.p[0]), pr<u + 2>(d.p[0]), pr<u + 10>(d.p[0])};
        } else {
            constexpr int u = 4 * h;
            r = u32x4_t{pr<u>(d.p[0]), pr<u>(d.p[1]), pr<u + 2>(d.p[0]), pr<u + 2>(d.p[1])};
        }
        return __builtin_bit_cast(half8_t, r);
    }
    template <int u>
    __device__ __forceinline__ static uint32_t pr(const Period<K>& P) {
        return cb_pair<CB>(P.template state<u>(), P.template state<u + 1>());
    }

    // byte offset of this lane's A elements within a row (fp16, chunk 0, fragment 0)
    __device__ __forceinline__ static uint32_t a_lane_off() {
        const int q = lane_id() >> 4;
        return F8 ? 32u * krow(q) : 32u * (q >> 1) + 8u * (q & 1);
    }
    // A fragment f at row byte offset off (row start + a_lane_off) of the chunk at byte k0
    template <int f, typename R>
    __device__ __forceinline__ static half8_t load_a(R rsrc, uint32_t off, int k0) {
        if constexpr (F8) {
            return __builtin_bit_cast(half8_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)(off + 16 * f), k0, 0));
        } else {
            const auto lo = __builtin_amdgcn_raw_buffer_load_b64(rsrc, (int)(off + 64 * f), k0, 0);
            const auto hi = __builtin_amdgcn_raw_buffer_load_b64(rsrc, (int)(off + 64 * f + 16), k0, 0);
            return __builtin_bit_cast(half8_t, u32x4_t{lo[0], lo[1], hi[0], hi[1]});
        }
    }
    // column of accumulator (column pair cc, half h) in the wave's 64 columns, for this lane
    __device__ __forceinline__ static int col(int cc, int h) {
        const int n = lane_id() & 15;
        return 16 * (2 * cc + (n >> 3)) + 8 * h + (n & 7);
    }
};

constexpr uint32_t kOob = 0x80000000u;            // a byte offset outside every descriptor used here (< 2 GiB each)

// acc[b][cc][h] += A[16 b .. 16 b + 15][chunks c0 .. c1) x W[chunks][64 columns]. ra / aoff: descriptor and per-block
// row byte offsets (kOob: a row that reads zero) of A, rows of fp16; rw / woff: descriptor and lane offset of the
// trellis strip. The words of PD chunks and the A fragments of one chunk are in flight while a chunk is decoded.
template <int K, int NB, bool NAT, int CB, typename R>
__device__ __forceinline__ void regb_core(R rw, uint32_t woff, int tiles_n, R ra, const uint32_t (&aoff)[NB], int c0,
                                          int c1, float4_t (&acc)[NB][2][2]) {
    using B = RegB<K, NAT, CB>;
    constexpr int PD = B::NW <= 6 ? 4 : 3;
    const uint32_t cb = B::chunk_bytes(tiles_n);
    const int src = B::prev_lane();
    uint32_t wd[PD][B::NW];
    half8_t a[2][NB];
#pragma unroll
    for (int j = 0; j < PD; ++j) B::load(wd[j], rw, c0 + j < c1 ? woff + (uint32_t)(c0 + j) * cb : kOob, tiles_n);
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        a[0][b] = B::template load_a<0>(ra, aoff[b], c0 * 128);
        a[1][b] = B::template load_a<1>(ra, aoff[b], c0 * 128);
    }
    for (int c = c0; c < c1; c += PD) {
#pragma unroll
        for (int j = 0; j < PD; ++j) {
            if (c + j >= c1) break;
            const int kn = min(c + j + 1, c1 - 1) * 128;               // the next chunk's A (the last one's again)
            typename B::Dec d[2];
            B::arrange(wd[j]);
            auto half = [&](auto F) {
                constexpr int f = decltype(F)::value;
                if (B::F8 ? f == 0 : true) {
                    B::prep(d[0], wd[j], B::F8 ? 0 : f, 0, src);
                    B::prep(d[1], wd[j], B::F8 ? 0 : f, 1, src);
                }
#pragma unroll
                for (int cc = 0; cc < 2; ++cc) {
                    const half8_t b0 = B::template frag<f, 0>(d[cc]), b1 = B::template frag<f, 1>(d[cc]);
#pragma unroll
                    for (int b = 0; b < NB; ++b) {
                        acc[b][cc][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[f][b], b0, acc[b][cc][0], 0, 0, 0);
                        acc[b][cc][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[f][b], b1, acc[b][cc][1], 0, 0, 0);
                    }
                }
#pragma unroll
                for (int b = 0; b < NB; ++b) a[f][b] = B::template load_a<f>(ra, aoff[b], kn);
            };
            half(std::integral_constant<int, 0>{});
            half(std::integral_constant<int, 1>{});
            B::load(wd[j], rw, c + j + PD < c1 ? woff + (uint32_t)(c + j + PD) * cb : kOob, tiles_n);
        }
    }
}

// A rows of a K chunk in LDS: row r at 128 r, its 16-byte piece j in slot j ^ ((r >> 1) & 7), so that the pieces of a
// staging store and 8 consecutive rows of a fragment read fall on distinct banks. A ds_read_b128 serves the 8-lane blocks
// (0, 3), (1, 2), (4, 7) and (5, 6) of the wave together (measured with a probe), i.e. rows 0-7 of one k-group with rows 8-15
// of its neighbour: distinct banks if both k-groups' pieces are in one half of the eight. They are but for the swapped words
// of K = 3 (tile-rows 0, 2, 1, 3), whose reads take two passes; whole layers do not show it (8,192 tokens 1,080-1,093 us so,
// 1,091-1,095 us with the tile-rows in order and half lines loaded). For V < 32 the two pieces of a tile-row are
// stored regrouped ({lo, lo}, {hi, hi}), so that a fragment is one 16-byte read for every K.
__device__ __forceinline__ uint32_t a_slot16(int r, int j) { return (uint32_t)(r * 128 + ((j ^ ((r >> 1) & 7)) << 4)); }

// The same product with the A rows staged through LDS for the WV waves of a workgroup (64 columns each), for more rows:
// NPROJ matrices of 16 NB rows (wave's matrix: proj), double-buffered, one barrier per chunk. Thread unit i covers 32
// bytes of one row of one matrix: soff[i] its byte offset in ra (kOob reads zeros). SD chunks of A are in flight in
// registers ahead of their LDS stores. PF > 0: PF fragments of A are read ahead of their MFMAs, the first ones before the
// chunk's decode (where the accumulators leave the registers for them).
template <int NB, int WV, int NPROJ>
struct AUnits {
    static constexpr int N = NPROJ * 16 * NB * 4;    // 32-byte units of a chunk
    static constexpr int NU = (N + 64 * WV - 1) / (64 * WV);
    __device__ __forceinline__ static int index(int i) { return (int)threadIdx.x + i * 64 * WV; }
    __device__ __forceinline__ static bool live(int i) { return N % (64 * WV) == 0 || index(i) < N; }
    __device__ __forceinline__ static int proj(int i) { return (index(i) >> 2) / (16 * NB); }
    __device__ __forceinline__ static int row(int i) { return (index(i) >> 2) % (16 * NB); }
    static constexpr int kBuf = NPROJ * 16 * NB * 128;
};

template <int K, int NB, int WV, int NPROJ, bool NAT, int CB, int SD, int PF, typename R>
__device__ __forceinline__ void regb_lds_core(R rw, uint32_t woff, int tiles_n, R ra,
                                              const uint32_t (&soff)[AUnits<NB, WV, NPROJ>::NU], int nch, int proj,
                                              uint8_t* lds, float4_t (&acc)[NB][2][2]) {
    using B = RegB<K, NAT, CB>;
    using U = AUnits<NB, WV, NPROJ>;
    constexpr int PD = NB <= 4 && B::NW <= 8 ? 4 : 2;
    static_assert(PD % 2 == 0 && PD % SD == 0, "buffer and register indices are compile-time within PD chunks");
    const uint32_t cb = B::chunk_bytes(tiles_n);
    const int src = B::prev_lane(), l = lane_id(), q = l >> 4;
    uint32_t wd[PD][B::NW];
    u32x4_t st[SD][U::NU][2];
    auto stage_load = [&](int s, int c) {        // (past the last chunk: the last one again)
#pragma unroll
        for (int i = 0; i < U::NU; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
                st[s][i][j] = __builtin_bit_cast(
                    u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(ra, (int)(soff[i] + 16 * j), min(c, nch - 1) * 128, 0));
    };
    auto stage_store = [&](int s, int buf) {
#pragma unroll
        for (int i = 0; i < U::NU; ++i)
            if (U::live(i)) {
                uint8_t* p = lds + buf * U::kBuf + U::proj(i) * (16 * NB * 128);
                const int r = U::row(i), j = 2 * (U::index(i) & 3);
                const u32x4_t lo = st[s][i][0], hi = st[s][i][1];
                if constexpr (B::F8) {
                    *(u32x4_t*)(p + a_slot16(r, j)) = lo;
                    *(u32x4_t*)(p + a_slot16(r, j + 1)) = hi;
                } else {
                    *(u32x4_t*)(p + a_slot16(r, j)) = u32x4_t{lo[0], lo[1], hi[0], hi[1]};
                    *(u32x4_t*)(p + a_slot16(r, j + 1)) = u32x4_t{lo[2], lo[3], hi[2], hi[3]};
                }
            }
    };
#pragma unroll
    for (int j = 0; j < SD; ++j) stage_load(j, j);
#pragma unroll
    for (int j = 0; j < PD; ++j) B::load(wd[j], rw, j < nch ? woff + (uint32_t)j * cb : kOob, tiles_n);
    stage_store(0, 0);
    stage_load(0, SD);
    __syncthreads();
    const uint8_t* ab = lds + proj * (16 * NB * 128);
    for (int c = 0; c < nch; c += PD) {
#pragma unroll
        for (int j = 0; j < PD; ++j) {
            if (c + j >= nch) break;
            if (c + j + 1 < nch) stage_store((j + 1) % SD, (j + 1) & 1);
            stage_load((j + 1) % SD, c + j + 1 + SD);
            const uint8_t* a0 = ab + (j & 1) * U::kBuf;
            typename B::Dec d[2];
            B::arrange(wd[j]);
            auto half = [&](auto F) {
                constexpr int f = decltype(F)::value;
                if (B::F8 ? f == 0 : true) {
                    B::prep(d[0], wd[j], B::F8 ? 0 : f, 0, src);
                    B::prep(d[1], wd[j], B::F8 ? 0 : f, 1, src);
                }
                const uint8_t* af = a0 + a_slot16(l & 15, B::F8 ? 2 * B::krow(q) + f : 4 * f + q);
                auto rd = [&](int b) { return *(const half8_t*)(af + b * 16 * 128); };
                constexpr int kPf = PF > 0 ? PF : 1;
                half8_t w[2][2], a[kPf];
                if constexpr (PF > 0) {          // before the decode, so that it covers their latency
#pragma unroll
                    for (int b = 0; b < PF; ++b) a[b] = rd(b);
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int cc = 0; cc < 2; ++cc) {
                    w[cc][0] = B::template frag<f, 0>(d[cc]);
                    w[cc][1] = B::template frag<f, 1>(d[cc]);
                }
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    const half8_t ab16 = PF > 0 ? a[b % kPf] : rd(b);
#pragma unroll
                    for (int cc = 0; cc < 2; ++cc)
#pragma unroll
                        for (int h = 0; h < 2; ++h)
                            acc[b][cc][h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ab16, w[cc][h], acc[b][cc][h], 0, 0, 0);
                    if (PF > 0 && b + PF < NB) {
                        a[b % kPf] = rd(b + PF);
                        __builtin_amdgcn_sched_group_barrier(0x8, 4, 0);
                        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    }
                }
            };
            half(std::integral_constant<int, 0>{});
            half(std::integral_constant<int, 1>{});
            B::load(wd[j], rw, c + j + PD < nch ? woff + (uint32_t)(c + j + PD) * cb : kOob, tiles_n);
            __syncthreads();
        }
    }
}

}  // namespace exl3
