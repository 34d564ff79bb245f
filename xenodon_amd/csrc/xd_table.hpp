// The start table: which cell holds which place, and what its entry says.  For
// the kernels and for the host's check of them.
#pragma once

#include <hip/hip_runtime.h>

#include "xd_internal.hpp"

namespace xd {

// Index in the start table of the cell at position bits (x, y, z): 4x4x4 cells
// together, 512 B, as the rays of a tile walk neighbouring cells along any axis.
__host__ __device__ __forceinline__ uint32_t table_cell(uint32_t x, uint32_t y, uint32_t z) {
    constexpr uint32_t sh = 23u - kTableLevel, b = kTableLevel - 2;
    return ((z >> (sh + 2)) << (2 * b) | (y >> (sh + 2)) << b | (x >> (sh + 2))) << 6 | (z >> sh & 3u) << 4 |
           (y >> sh & 3u) << 2 | (x >> sh & 3u);
}
// Its inverse: the position bits of a cell's lower corner.
__host__ __device__ __forceinline__ uint3 table_place(uint32_t cell) {
    constexpr uint32_t sh = 23u - kTableLevel, b = kTableLevel - 2, m = (1u << b) - 1u;
    return make_uint3((cell >> 6 & m) << (sh + 2) | (cell & 3u) << sh,
                      (cell >> (b + 6) & m) << (sh + 2) | (cell >> 2 & 3u) << sh,
                      (cell >> (2 * b + 6) & m) << (sh + 2) | (cell >> 4 & 3u) << sh);
}

// Entry `i` of a table whose cells are coarser by `shift` levels: its index in the
// table's memory (*at) and what it holds, the walk of build_start_table.  False from
// the number of such cells on.  rec: the internal nodes' records, or null.
__host__ __device__ __forceinline__ bool table_entry(const uint32_t* cw, uint32_t root_tag, uint32_t index_mask,
                                                     uint32_t shift, const uint4* rec, uint32_t i, uint32_t* at,
                                                     uint2* entry) {
    const uint32_t levels = kTableLevel - shift;
    uint3 p = table_place(i);
    *at = i;
    if (shift) {  // the cells below 2^levels of each axis
        const uint32_t m = (1u << levels) - 1u, sh = 23u - levels;
        if (i >> (3 * levels)) return false;
        p = make_uint3((i & m) << sh, (i >> levels & m) << sh, (i >> (2 * levels) & m) << sh);
        *at = table_cell(p.x >> shift, p.y >> shift, p.z >> shift);
    }
    uint32_t word = root_tag, level = 0;
    while (!(word & kTagLeaf) && level < levels) {
        const uint32_t s = 22u - level;
        const uint32_t k = (p.x >> s & 1u) << 2 | (p.y >> s & 1u) << 1 | (p.z >> s & 1u);
        word = cw[(uint64_t)(word & index_mask) * 8 + k];
        ++level;
    }
    if (!(word & kTagLeaf) && rec && (rec[(uint64_t)(word & index_mask) * (kRecWords / 4)].y & 0xFFu) == 0)
        level |= kTableLowNode;
    *entry = make_uint2(word, level);
    return true;
}

}  // namespace xd
