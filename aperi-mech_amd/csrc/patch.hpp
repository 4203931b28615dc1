// Node patches (see patch.hip): what the step and the reverse step share.
#pragma once

#include "element.hpp"
#include "internal.hpp"

namespace aphip {

constexpr uint16_t kNewTile = 0x8000;   // entry flag: the node's first element of another tile
constexpr int kBatch = 8;               // entries of a node are padded to a multiple of this

// rows between the slot blocks of the force rows (as in the tile kernel: the slots of one
// element sit 24 banks apart)
__host__ __device__ __forceinline__ int patch_stride(int n) { return n + ((4 - n) & 31); }

// force row of (local element, slot), in rows of three doubles: Tet4 slot-major, Hex8 in the
// element's LDS row
__host__ __device__ __forceinline__ int force_row(int npe, int epad, int le, int k) {
    return npe == 4 ? k * patch_stride(epad) + le : (kHexRow / 3) * le + k;
}

// Component d's sum of a node's force rows (F: rows + d), pk: its (start << 16) | count.  The
// sums stay in order, grouped by tile, and the LDS latency is paid once per kBatch entries.
__device__ __forceinline__ double patch_sum(const double *F, const uint16_t *entries, uint32_t pk) {
    const int st = (int)(pk >> 16) * kBatch, cnt = (int)(pk & 0xffffu);
    double f = 0.0, t = 0.0;
    for (int j = 0; j < cnt; j += kBatch) {
        const uint4 w = *reinterpret_cast<const uint4 *>(entries + st + j);
        const unsigned en[kBatch] = {w.x & 0xffffu, w.x >> 16, w.y & 0xffffu, w.y >> 16,
                                     w.z & 0xffffu, w.z >> 16, w.w & 0xffffu, w.w >> 16};
        double r[kBatch];
#pragma unroll
        for (int q = 0; q < kBatch; ++q) r[q] = F[3 * (en[q] & 0x7fffu)];
#pragma unroll
        for (int q = 0; q < kBatch; ++q) {
            const bool fresh = en[q] & kNewTile;
            f = fresh ? f + t : f;
            t = fresh ? 0.0 : t;
            t = j + q < cnt ? t + r[q] : t;
        }
    }
    return f + t;
}

}  // namespace aphip
