// The misses of a cached call that the grouped expert kernels serve, copied from host memory into their new slots beside
// those kernels' own work (reference: the write-through and victim write-back of a8:371-395, 1168-1189).
//
// PCIe bounds these copies (1.2 MB per expert of H 2048 / I 512 / K 3 are 22 us at 53 GB/s), so the layer must not stand
// still behind them: the first workgroups of the sort-and-Hadamard launch copy what gate/up reads, those of the gate/up
// launch copy the down trellis, each piece of a victim leaves the slot right before its successor arrives, so that both
// PCIe directions are in use, and the combine launch commits the table. With victims, fills and commit as launches of
// their own before the products, and now (us, 3 layers): 16 rows of uniform routing, 95 % of the experts in slots 277,
// now 230-237 (the fused decode kernel: 252); 90 % 437, now 390-401 (433); every pick in its slot 75.5, now 72.3 (122).
// Tiered decode of 48 layers at 16 rows 3,309, now 3,632 tok/s.
#pragma once
#include "exl3_common.cuh"
#include "exl3_kernels.h"

namespace exl3 {

typedef uint32_t u32x4_f __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(1))) u32x4_f gfill_t;

// groups of 256 threads that copy, of a launch: more in flight reads host memory slower (16 rows as above, 95 %: 32 / 64 /
// 128 / 256 groups 254 / 231 / 239 / 242 us)
constexpr int kFillWorkers = 64;
constexpr int kFillUnit = 256 * 16;              // bytes that a group has in flight
__host__ __device__ constexpr int fill_workgroups(int threads) { return kFillWorkers / (threads / 256); }

// the share of workgroup wg (of fill_workgroups(NT)) of part 0: gate/up trellis and scales (to the end of the victim's
// slot, which may hold a larger expert), or of part 1: down trellis. Every group takes one run of all the misses' units.
template <int NT>
__device__ __forceinline__ void fill_part(const GroupedArgs& A, int part, int wg) {
    const FillArgs& F = A.f;
    const int64_t gu = A.g.gu_bytes, dn = A.g.d_bytes, blob = A.g.blob;
    const int64_t end = F.vict && F.sstride > blob ? F.sstride : blob;
    auto units = [](int64_t n) { return (int)((n + kFillUnit - 1) / kFillUnit); };
    const int ugu = units(gu), nu = part ? units(dn) : ugu + units(end - gu - dn), t16 = threadIdx.x % 256 * 16;
    const int64_t all = (int64_t)F.list[0] * nu, w = wg * (NT / 256) + threadIdx.x / 256;
    int64_t it = all * w / kFillWorkers;
    const int64_t last = all * (w + 1) / kFillWorkers;
    while (it < last) {
        const int mi = (int)(it / nu), u0 = (int)(it - (int64_t)mi * nu), e = F.list[1 + mi];
        const int u1 = (int)min((int64_t)nu, last - (int64_t)mi * nu);
        const uint8_t* src = (const uint8_t*)F.ptrs[e];
        uint8_t* slot = (uint8_t*)F.fill[e];
        uint8_t* rec = nullptr;                  // the victim's record (none: an empty slot, or a valid copy there)
        if (F.vict && F.vict[1 + 2 * mi] >= 0) {
            const int old = F.vict[1 + 2 * mi];
            rec = (uint8_t*)(F.vaddr ? F.vaddr[mi] : F.host_base[old / A.E] + (int64_t)(old % A.E) * F.hstride);
            if (F.ram_res && part == 0 && u0 == 0 && t16 == 0) F.ram_res[old] = 1;
        }
        for (int u = u0; u < u1; ++u) {          // sections [0, gu), [gu + dn, end) or [gu, gu + dn)
            const int64_t o = (part ? gu : u < ugu ? 0 : gu + dn) + (int64_t)(part || u < ugu ? u : u - ugu) * kFillUnit + t16;
            const int64_t hi = part ? gu + dn : u < ugu ? gu : end;
            const bool out = rec && o < min(hi, F.sstride), in = o < min(hi, blob);
            u32x4_f v{}, f{};
            if (out) v = *(const gfill_t*)(uintptr_t)(slot + o);
            if (in) f = *(const gfill_t*)(uintptr_t)(src + o);
            if (out) *(gfill_t*)(uintptr_t)(rec + o) = v;
            if (in) *(gfill_t*)(uintptr_t)(slot + o) = f;
        }
        it += u1 - u0;
    }
}

}  // namespace exl3
