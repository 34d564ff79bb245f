// Host check of the start table as the device has it (csrc/xd_table.hpp), against
// build_start_table's plain form.  Usage: table_check <nodes.words> <wide 0|1>
// For shift 0 and the one of the tree's depth:
//   * table_cell and table_place are each other's inverse;
//   * the entries take each cell of the coarser grid once, and no place has an entry
//     other than the one that the plain table has for any cell of it;
//   * kTableLowNode is set where, and only where, the node has no internal children.
// Prints "ok" and exits 0, or prints the first failures and exits 1.
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "xd_runtime.hpp"
#include "xd_table.hpp"

using namespace xd;

static int failures = 0;
#define CHECK(cond, ...)                     \
    do {                                     \
        if (!(cond) && failures++ < 10) {    \
            std::printf("FAIL %s: ", #cond); \
            std::printf(__VA_ARGS__);        \
            std::printf("\n");               \
        }                                    \
    } while (0)

static uint32_t height(const std::vector<uint32_t>& w, uint32_t i) {
    if (w[(uint64_t)i * kNodeWords + 9] & kLeafMask) return 0;
    uint32_t h = 0;
    for (int k = 0; k < 8; ++k) h = std::max(h, height(w, w[(uint64_t)i * kNodeWords + k]));
    return h + 1;
}

int main(int argc, char** argv) {
    if (argc != 3) return 2;
    FILE* f = std::fopen(argv[1], "rb");
    if (!f) return 2;
    std::vector<uint32_t> w;
    uint32_t buf[4096];
    size_t r;
    while ((r = std::fread(buf, 4, 4096, f)) > 0) w.insert(w.end(), buf, buf + r);
    std::fclose(f);
    const uint64_t n = w.size() / kNodeWords;
    const bool wide = std::atoi(argv[2]) != 0;
    std::vector<uint32_t> cw(n * 8), meta(n * 2);
    uint32_t top[kTopLevels], empty_start = 0, leaf_base = 0;
    build_tagged_layout(w.data(), n, cw.data(), meta.data(), top, wide, false, &empty_start, &leaf_base);
    const uint32_t mask = wide ? kWideIndexMask : kIndexMask, empty_tag = wide ? 0u : kTagEmpty;
    const uint32_t root_tag = (w[9] & kLeafMask) ? (kTagLeaf | ((w[8] & 0xFFFFFFu) ? 0u : empty_tag)) : 0u;
    std::vector<uint2> plain(kTableCells);
    build_start_table(cw.data(), root_tag, mask, plain.data());
    // what a record's second word says of a node's internal children
    std::vector<uint4> rec(n * (kRecWords / 4), make_uint4(0, 0, 0, 0));
    for (uint64_t i = 0; i < n; ++i) {
        if (meta[i * 2 + 1] & kLeafMask) continue;
        for (uint32_t k = 0; k < 8; ++k)
            if (!(cw[i * 8 + k] & kTagLeaf)) rec[i * (kRecWords / 4)].y |= 1u << k;
    }
    const uint32_t depth = height(w, 0), most = table_shift_of(depth);
    CHECK(most == (depth < kTableLevel ? kTableLevel - depth : 0), "shift %u of depth %u", most, depth);
    for (uint32_t i = 0; i < kTableCells; ++i) {
        const uint3 p = table_place(i);
        CHECK(table_cell(p.x, p.y, p.z) == i, "cell %u", i);
    }
    uint64_t low = 0;
    for (uint32_t shift = 0; shift <= most; shift += std::max(most, 1u)) {
        const uint32_t levels = kTableLevel - shift;
        std::vector<uint2> table(kTableCells, make_uint2(0xDEADBEEFu, 0));
        std::vector<uint8_t> set(kTableCells, 0);
        uint64_t count = 0;
        for (uint32_t i = 0; i < kTableCells; ++i) {
            uint32_t at = 0;
            uint2 e;
            if (!table_entry(cw.data(), root_tag, mask, shift, rec.data(), i, &at, &e)) break;
            CHECK(at < kTableCells && !set[at], "shift %u entry %u at %u", shift, i, at);
            if (at >= kTableCells) break;
            set[at] = 1;
            table[at] = e;
            ++count;
        }
        CHECK(count == 1ull << (3 * levels), "shift %u: %llu entries", shift, (unsigned long long)count);
        constexpr uint32_t sh = 23u - kTableLevel;
        for (uint32_t z = 0; z < 1u << kTableLevel; ++z)
            for (uint32_t y = 0; y < 1u << kTableLevel; ++y)
                for (uint32_t x = 0; x < 1u << kTableLevel; ++x) {
                    const uint2 want = plain[((uint64_t)z << (2 * kTableLevel)) | (y << kTableLevel) | x];
                    // the last place of the cell: its low bits must not matter
                    const uint32_t in = (1u << sh) - 1u;
                    const uint2 e = table[table_cell((x << sh | in) >> shift, (y << sh | in) >> shift,
                                                     (z << sh | in) >> shift)];
                    const bool leaf = (want.x & kTagLeaf) != 0;
                    const bool is_low = !leaf && (rec[(uint64_t)(want.x & mask) * (kRecWords / 4)].y & 0xFFu) == 0;
                    low += is_low;
                    CHECK(e.x == want.x && (e.y & kTableLevelMask) == want.y && ((e.y & kTableLowNode) != 0) == is_low,
                          "shift %u cell (%u, %u, %u): {%08x, %x}, want {%08x, %x, low %d}", shift, x, y, z, e.x, e.y,
                          want.x, want.y, (int)is_low);
                }
    }
    if (failures) {
        std::printf("%d failures\n", failures);
        return 1;
    }
    std::printf("ok: depth %u, shift %u, low cells %d\n", depth, most, low ? 1 : 0);
    return 0;
}
