// Device layout of an octree derived on the GPU from the .svo nodes (the
// layout itself: xd_layout.cpp), and the start table.
//
// The numbering that a recursive walk gives comes from two prefix sums here.
// The converter writes a tree in reverse post-order (OctreeConstruction.h:
// 92-112), a depth-first order from the root, so sibling groups taken in the
// order of their parents' old indices are depth-first too.  Within each class
// of the final order (internal nodes, leaves with colour, empty leaves) a
// child's index is then the number of that class's children of all earlier
// parents, plus those before it among its siblings.  The parents of the top
// levels, numbered breadth-first, come first; the host walks those few.
//
// Three passes over the nodes, one thread a node, blocks of kOctBlock:
//   k_oct_classify  checks the node, looks at its children's classes, sums
//                   them per block
//   k_oct_number    scans the block's sums, gives each child its word
//   k_oct_emit      scans again (cheaper than keeping 12 bytes a node) and
//                   writes child words, records, colours, depths and ropes
// The passes read the nodes' 40 bytes and, scattered over nearby nodes, their
// children's words: for a tree of 1.3 million nodes (192x137x192 voxels) 59 us
// with the checks, 24 and 30 us, about 1 TB/s each, then 53 us for the 128 MiB
// table (2.5 TB/s of stores, eight dependent loads a cell).  The host's
// derivation and uploads took 90 ms; a load from host memory went from 93 to
// 4.3 ms, of which the nodes' upload is 2.
//
// A tree is derived here if its nodes come in an order with children after
// their parent, each named once, and its internal nodes' depth fields are their
// depths: what the converter writes for sparse and rope trees.  DAGs, other
// orders, malformed trees (which the host path reports) and trees that leave no
// device memory for the nodes' copy are derived on the host.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "xd_runtime.hpp"
#include "xd_table.hpp"

namespace xd {
namespace {

constexpr uint32_t kOctBlock = 512;
constexpr uint32_t kTopParent = 0x80000000u;  // in a node's mask word: numbered with the top levels, slot in bits 20..27
constexpr uint32_t kMaxTopParents = 1 + 8 + 64;

struct OctFlags {
    uint32_t refused;      // malformed, out of order, or depth fields inexact
    uint32_t ropes;        // a leaf has a rope other than 0
    uint32_t inner_depth;  // largest depth field of an internal node
    uint32_t depth;        // ... of any node
    uint32_t total[4];     // children by class, parents of the top levels left out; internal nodes
    uint32_t twice;        // a node is named by two child words
    uint32_t bad_rope;     // a leaf's rope or depth field is not the tree's
};

// First index of each class, for the nodes that the prefix sums number and
// overall.
struct OctBases {
    uint32_t after_top[3];  // children of top-level parents, by class (the root counts as class 0)
    uint32_t leaf_base, empty_base;
};

// Classes of a parent's children: bits 0..7 internal, 8..15 leaf with colour.
__device__ __forceinline__ uint32_t inner_mask(uint32_t m) { return m & 0xFFu; }
__device__ __forceinline__ uint32_t colour_mask(uint32_t m) { return (m >> 8) & 0xFFu; }
// A thread's share of its block's sums: children by class, 16 bits each, and
// whether it is a parent.  512 threads of 8 children stay below 2^16.
__device__ __forceinline__ uint64_t counts_of(uint32_t m, bool inner) {
    if (!inner) return 0;
    const uint64_t one = 1ull << 48;
    if (m & kTopParent) return one;
    const uint32_t i = __popc(inner_mask(m)), c = __popc(colour_mask(m));
    return one | (uint64_t)i | (uint64_t)c << 16 | (uint64_t)(8 - i - c) << 32;
}

// Exclusive scan of v over the block; *total gets the block's sum.
__device__ uint64_t block_scan(uint64_t v, uint64_t* total) {
    __shared__ uint64_t wave_sum[kOctBlock / 64];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint64_t s = v;
#pragma unroll
    for (uint32_t d = 1; d < 64; d <<= 1) {
        const uint64_t o = __shfl_up((unsigned long long)s, d, 64);
        if (lane >= d) s += o;
    }
    if (lane == 63) wave_sum[wave] = s;
    __syncthreads();
    uint64_t before = 0, all = 0;
#pragma unroll
    for (uint32_t w = 0; w < kOctBlock / 64; ++w) {
        if (w < wave) before += wave_sum[w];
        all += wave_sum[w];
    }
    __syncthreads();  // the caller may scan again
    *total = all;
    return before + s - v;
}

__global__ void k_oct_init(uint32_t* masks, uint32_t* words, uint64_t n, OctFlags* flags) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) masks[i] = words[i] = 0;  // a node that nothing names keeps index 0, in bounds
    if (i < sizeof(OctFlags) / 4) reinterpret_cast<uint32_t*>(flags)[i] = 0;
}

// top: {old index, first child of each class} of the top-level parents.
__global__ void k_oct_mark_top(const uint4* top, uint32_t count, uint32_t* masks) {
    const uint32_t s = threadIdx.x;
    if (s < count) masks[top[s].x] = kTopParent | (s << 20);
}

__device__ __forceinline__ void load_node(const uint2* raw, uint64_t i, uint32_t c[8]) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint2 v = raw[i * 5 + k];
        c[2 * k] = v.x;
        c[2 * k + 1] = v.y;
    }
}

__global__ __launch_bounds__(kOctBlock) void k_oct_classify(const uint2* __restrict__ raw, uint32_t n,
                                                            uint32_t* __restrict__ masks, OctFlags* flags,
                                                            uint64_t* __restrict__ sums) {
    const uint64_t i = (uint64_t)blockIdx.x * kOctBlock + threadIdx.x;
    bool refused = false, ropes = false, inner = false;
    uint32_t depth = 0, m = 0;
    if (i < n) {
        uint32_t c[8];
        load_node(raw, i, c);
        const uint32_t ld = raw[i * 5 + 4].y;
        depth = ld & kDepthMask;
        inner = !(ld & kLeafMask);
        refused = depth > 64u || (i == 0 && inner && depth != 0);
        for (int k = 0; k < 8; ++k) refused |= c[k] >= n;
        if (!refused) {
            if (inner) {
                m = masks[i];
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const uint2 cm = raw[(uint64_t)c[k] * 5 + 4];  // {colour, is_leaf_depth}
                    refused |= c[k] <= i;
                    if (!(cm.y & kLeafMask)) {
                        m |= 1u << k;
                        refused |= (cm.y & kDepthMask) != depth + 1u;
                    } else if (cm.x & 0xFFFFFFu) {
                        m |= 0x100u << k;
                    }
                }
                masks[i] = m;
            } else {
#pragma unroll
                for (int k = 0; k < 6; ++k) ropes |= c[k] != 0;
            }
        }
    }
    uint64_t total;
    block_scan(counts_of(m, inner), &total);
    if (threadIdx.x == 0) sums[blockIdx.x] = total;
    __shared__ uint32_t s_inner, s_depth, s_refused, s_ropes;
    if (threadIdx.x == 0) s_inner = s_depth = s_refused = s_ropes = 0;
    __syncthreads();
    if (inner) atomicMax(&s_inner, depth);
    atomicMax(&s_depth, depth);
    if (refused) s_refused = 1;
    if (ropes) s_ropes = 1;
    __syncthreads();
    if (threadIdx.x == 0) {  // most blocks find the flags already there
        if (s_inner > flags->inner_depth) atomicMax(&flags->inner_depth, s_inner);
        if (s_depth > flags->depth) atomicMax(&flags->depth, s_depth);
        if (s_refused && !flags->refused) atomicOr(&flags->refused, 1u);
        if (s_ropes && !flags->ropes) atomicOr(&flags->ropes, 1u);
    }
}

// Exclusive scan of the blocks' sums, one block: base[b] = {by class, 0}.
__global__ __launch_bounds__(kOctBlock) void k_oct_scan(const uint64_t* __restrict__ sums, uint32_t blocks,
                                                        uint4* __restrict__ base, OctFlags* flags) {
    __shared__ uint32_t part[4][kOctBlock / 64];
    uint32_t run[4] = {0, 0, 0, 0};
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    for (uint32_t b0 = 0; b0 < blocks; b0 += kOctBlock) {
        const uint32_t b = b0 + threadIdx.x;
        const uint64_t v = b < blocks ? sums[b] : 0;
        uint32_t mine[4], s[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            mine[q] = s[q] = (uint32_t)(v >> (16 * q)) & 0xFFFFu;
            for (uint32_t d = 1; d < 64; d <<= 1) {
                const uint32_t o = __shfl_up(s[q], d, 64);
                if (lane >= d) s[q] += o;
            }
            if (lane == 63) part[q][wave] = s[q];
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            uint32_t before = 0, all = 0;
            for (uint32_t w = 0; w < kOctBlock / 64; ++w) {
                if (w < wave) before += part[q][w];
                all += part[q][w];
            }
            s[q] = run[q] + before + s[q] - mine[q];
            run[q] += all;
        }
        if (b < blocks) base[b] = make_uint4(s[0], s[1], s[2], 0);
        __syncthreads();
    }
    if (threadIdx.x < 4) flags->total[threadIdx.x] = run[threadIdx.x];
}

// Final index of the first child of each class of the thread's node.
__device__ __forceinline__ void child_bases(uint32_t m, bool inner, const uint4* base, const uint4* top,
                                            const OctBases& B, uint32_t first[3]) {
    uint64_t total;
    const uint64_t s = block_scan(counts_of(m, inner), &total);
    const uint4 b = base[blockIdx.x];
    if (m & kTopParent) {
        const uint4 t = top[(m >> 20) & 0x7Fu];
        first[0] = t.y;
        first[1] = t.z;
        first[2] = t.w;
    } else {
        first[0] = B.after_top[0] + b.x + (uint32_t)(s & 0xFFFFu);
        first[1] = B.after_top[1] + b.y + (uint32_t)((s >> 16) & 0xFFFFu);
        first[2] = B.after_top[2] + b.z + (uint32_t)((s >> 32) & 0xFFFFu);
    }
    first[1] += B.leaf_base;
    first[2] += B.empty_base;
}

// Child k's final index, with its tags.
__device__ __forceinline__ uint32_t child_word(uint32_t m, const uint32_t first[3], uint32_t k, uint32_t empty_tag) {
    const uint32_t below = (1u << k) - 1u, im = inner_mask(m), cm = colour_mask(m);
    if (im >> k & 1u) return first[0] + __popc(im & below);
    if (cm >> k & 1u) return (first[1] + __popc(cm & below)) | kTagLeaf;
    return (first[2] + __popc(~(im | cm) & below)) | kTagLeaf | empty_tag;
}

// words[c]: the final word of every node; with depth_bits, the depth field in
// bits kRopeDepthShift.. (indices are below 2^25 then).
__global__ __launch_bounds__(kOctBlock) void k_oct_number(const uint2* __restrict__ raw, uint32_t n,
                                                          const uint32_t* __restrict__ masks,
                                                          const uint4* __restrict__ base, const uint4* __restrict__ top,
                                                          OctBases B, uint32_t root_tag, uint32_t empty_tag,
                                                          uint32_t depth_bits, uint32_t* __restrict__ words) {
    const uint64_t i = (uint64_t)blockIdx.x * kOctBlock + threadIdx.x;
    const bool inner = i < n && !(raw[i * 5 + 4].y & kLeafMask);
    const uint32_t m = inner ? masks[i] : 0;
    uint32_t first[3];
    child_bases(m, inner, base, top, B, first);
    if (i == 0) words[0] = root_tag | (depth_bits ? (raw[4].y & kDepthMask) << kRopeDepthShift : 0u);
    if (!inner) return;
    uint32_t c[8];
    load_node(raw, i, c);
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) {
        uint32_t w = child_word(m, first, k, empty_tag);
        if (depth_bits) w |= (raw[(uint64_t)c[k] * 5 + 4].y & kDepthMask) << kRopeDepthShift;
        words[c[k]] = w;
    }
}

__global__ __launch_bounds__(kOctBlock) void k_oct_emit(const uint2* __restrict__ raw, uint32_t n,
                                                        const uint32_t* __restrict__ masks,
                                                        const uint4* __restrict__ base, const uint4* __restrict__ top,
                                                        OctBases B, uint32_t empty_tag, uint32_t index_mask,
                                                        const uint32_t* __restrict__ words, uint32_t* __restrict__ cw,
                                                        uint4* __restrict__ rec, uint32_t* __restrict__ meta,
                                                        OctFlags* flags) {
    const uint64_t i = (uint64_t)blockIdx.x * kOctBlock + threadIdx.x;
    uint2 cm = make_uint2(0, kLeafMask);  // {colour, is_leaf_depth}
    if (i < n) cm = raw[i * 5 + 4];
    const bool inner = !(cm.y & kLeafMask);
    const uint32_t m = inner ? masks[i] : 0;
    uint32_t first[3];
    child_bases(m, inner, base, top, B, first);
    if (i >= n) return;
    const uint32_t id = words[i] & index_mask;
    meta[id] = cm.x;
    meta[(uint64_t)n + id] = cm.y;
    uint32_t c[8];
    load_node(raw, i, c);
    if (inner) {
        uint32_t w[8];
        bool twice = false;
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k) {
            w[k] = child_word(m, first, k, empty_tag);
            twice |= (words[c[k]] & index_mask) != (w[k] & index_mask);
        }
        if (twice) flags->twice = 1;
        uint4* const out = reinterpret_cast<uint4*>(cw + (uint64_t)id * 8);
        out[0] = make_uint4(w[0], w[1], w[2], w[3]);
        out[1] = make_uint4(w[4], w[5], w[6], w[7]);
        uint32_t low = 0;  // internal children without internal children
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k)
            if (inner_mask(m) >> k & 1u && inner_mask(masks[c[k]]) == 0) low |= 0x10000u << k;
        uint32_t col[8];  // 0 but for leaves with colour
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k)
            col[k] = colour_mask(m) >> k & 1u ? raw[(uint64_t)c[k] * 5 + 4].x & 0xFFFFFFu : 0u;
        uint4* const r = rec + (uint64_t)id * kRecWords / 4;
        r[0] = make_uint4(first[0], (m & 0xFFFFu) | low, 0, 0);
        r[1] = make_uint4(col[0], col[1], col[2], col[3]);
        r[2] = make_uint4(col[4], col[5], col[6], col[7]);
    } else if (id >= B.leaf_base) {  // six ropes; a leaf root has no planes
        const uint64_t nl = n - B.leaf_base, at = (uint64_t)B.leaf_base * 8 + (id - B.leaf_base);
#pragma unroll
        for (uint32_t k = 0; k < 6; ++k) cw[at + k * nl] = words[c[k]];
    } else {
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k) cw[k] = words[c[k]];
    }
}

// One cell of the start table a thread.
// stop: null, or a word that says, when set, that the child words are no tree's.
__global__ __launch_bounds__(256) void k_start_table(const uint32_t* __restrict__ cw, uint32_t root_tag,
                                                     uint32_t index_mask, uint32_t shift,
                                                     const uint4* __restrict__ rec, const uint32_t* stop,
                                                     uint2* __restrict__ table) {
    if (stop && *stop) return;
    uint32_t at;
    uint2 entry;
    if (table_entry(cw, root_tag, index_mask, shift, rec, blockIdx.x * 256 + threadIdx.x, &at, &entry)) table[at] = entry;
}

}  // namespace

// Whether the leaves' ropes lead where the tree's geometry says, so that a ray may
// go from leaf to leaf by position (fast_rope_cells).  A rope's target is the node
// beside the leaf at the leaf's level, or the leaf that holds that place; the table
// knows the place's leaf or its level-8 node, and whichever of the two is the
// higher must lead down to the other, in as many steps as there are levels between.
// A thread takes the leaves of one table cell: those above it if the cell is their
// first, else all below its node.  (A 1.3 M node load with its first frame, of which
// the rope walk is 0.1 ms less, 2.71 -> 2.75 ms.)
__global__ __launch_bounds__(256) void k_check_ropes(const uint32_t* __restrict__ cw, const uint32_t* __restrict__ meta,
                                                     uint32_t n, uint32_t leaf_base, uint32_t index_mask,
                                                     uint32_t depth, const uint2* __restrict__ table, OctFlags* flags) {
    if (flags->twice) return;  // no tree, and no table
    const uint32_t cell = blockIdx.x * 256 + threadIdx.x;
    const uint3 corner = table_place(cell);
    const uint2 own = table[cell];
    const uint32_t top = own.y & kTableLevelMask;
    if ((corner.x | corner.y | corner.z) & ((1u << (23u - top)) - 1u)) return;
    const auto step = [&](uint32_t word, uint32_t level, const uint32_t p[3]) {  // the child towards p
        const uint32_t s = 22u - level, k = (p[0] >> s & 1u) << 2 | (p[1] >> s & 1u) << 1 | (p[2] >> s & 1u);
        return cw[(uint64_t)(word & index_mask) * 8 + k];
    };
    // the leaves below own, by a counter of the cells of the finest level
    const uint32_t fine = own.x & kTagLeaf ? top : max(depth, top);
    for (uint32_t c = 0; c < 1u << 3 * (fine - top);) {
        uint32_t p[3] = {corner.x, corner.y, corner.z};
        uint32_t word = own.x, level = top;
        for (uint32_t b = 0; b < fine - top; ++b) {  // Morton order: three bits a level, the finest last
            const uint32_t o = c >> 3 * (fine - top - 1 - b) & 7u, s = 22u - top - b;
            p[0] |= (o >> 2 & 1u) << s;
            p[1] |= (o >> 1 & 1u) << s;
            p[2] |= (o & 1u) << s;
        }
        for (; !(word & kTagLeaf) && level < fine; ++level) word = step(word, level, p);
        c += 1u << 3 * (fine - level);
        const uint32_t leaf = word & index_mask, size = 1u << (23u - level);
        bool bad = !(word & kTagLeaf) || leaf < leaf_base || (meta[(uint64_t)n + leaf] & kDepthMask) != level;
        for (uint32_t k = 0; k < 6 && !bad; ++k) {
            uint32_t q[3] = {p[0], p[1], p[2]};
            q[k >> 1] += (k & 1u) ? 0u - size : size;
            const uint32_t rope = cw[(uint64_t)leaf_base * 8 + (uint64_t)k * (n - leaf_base) + (leaf - leaf_base)];
            if (q[k >> 1] >> 23) {
                bad = (rope & index_mask) != 0;
                continue;
            }
            const uint2 e = table[table_cell(q[0], q[1], q[2])];
            uint32_t at = e.y & kTableLevelMask, a = e.x, b = rope;
            if (at <= level) {  // from the table's node down to the leaf's level
                for (; at < level && !(a & kTagLeaf); ++at) a = step(a, at, q);
            } else {
                // from the rope's target, at the leaf's level, down to the table's node, each
                // level in between: a descendant of the target at the place's corner leads to
                // that node too, by fewer
                uint32_t l = level;
                for (; l < at && !(b & kTagLeaf); ++l) b = step(b, l, q);
                bad = l != at;
            }
            bad |= ((a ^ b) & index_mask) != 0;
        }
        if (bad) {
            flags->bad_rope = 1;
            return;
        }
    }
}

hipError_t launch_start_table(const uint32_t* cw, uint32_t root_tag, uint32_t index_mask, uint32_t shift, const uint4* rec,
                              const uint32_t* stop, uint2* table, hipStream_t s) {
    hipLaunchKernelGGL(k_start_table, dim3((uint32_t)(((kTableCells >> (3 * shift)) + 255) / 256)), dim3(256), 0, s, cw,
                       root_tag, index_mask, shift, rec, stop, table);
    return hipGetLastError();
}

bool derive_layout_on_device(xd_volume* v, const uint32_t* w, uint64_t n, bool wide) {
    // the top levels, breadth-first: {old index, first child of each class}
    std::vector<uint4> top;
    std::vector<uint32_t> level{0}, next;
    const bool root_leaf = (w[9] & kLeafMask) != 0;
    uint32_t count[3] = {1, 0, 0};  // nodes of the top levels so far, by class; the root is class 0
    if (n % 8 != 1 || (root_leaf && n != 1)) return false;  // no tree has so many nodes (most DAGs do)
    v->top[0] = 1;
    for (uint32_t L = 1; L < kTopLevels; ++L) {
        next.clear();
        for (uint32_t old : level) {
            const uint32_t* nd = w + (uint64_t)old * kNodeWords;
            if (nd[9] & kLeafMask) continue;
            // named twice, its children would be counted twice and the indices run past the nodes
            for (const uint4& t : top)
                if (t.x == old) return false;
            top.push_back(make_uint4(old, count[0], count[1], count[2]));
            for (int k = 0; k < 8; ++k) {
                if (nd[k] >= n) return false;
                const uint32_t* cn = w + (uint64_t)nd[k] * kNodeWords;
                ++count[!(cn[9] & kLeafMask) ? 0 : (cn[8] & 0xFFFFFFu) ? 1 : 2];
                next.push_back(nd[k]);
            }
        }
        if (top.size() > kMaxTopParents) return false;
        level.swap(next);
        v->top[L] = count[0];
    }
    hipStream_t s = v->ctx->stream;
    const uint32_t blocks = (uint32_t)((n + kOctBlock - 1) / kOctBlock);
    // The volume is one allocation: child words and records | colours and depths |
    // start table | flags.  The table is written last, and until then, where it is
    // large enough, it holds what the derivation needs for itself: nodes | masks |
    // words | block sums | block bases | top parents.  (A release costs 0.33 ms
    // from 128 MB on: with five allocations a load spent 0.8 of 3.1 ms on them.)
    const auto align = [](uint64_t b) { return (b + 255) & ~255ull; };
    const uint64_t at_masks = align(n * kNodeWords * 4), at_words = at_masks + align(n * 4),
                   at_sums = at_words + align(n * 4), at_base = at_sums + align(blocks * 8ull),
                   at_top = at_base + align(blocks * 16ull), tmp_bytes = at_top + align(kMaxTopParents * sizeof(uint4));
    const uint64_t at_meta = align(n * 8 * sizeof(uint32_t)), at_table = at_meta + align(n * 2 * sizeof(uint32_t)),
                   at_flags = at_table + kTableBytes;
    uint8_t *block = nullptr, *own = nullptr, *tmp = nullptr;
    OctFlags f{};
    hipError_t e = hipMalloc(&block, at_flags + 256);
    if (e == hipSuccess && tmp_bytes > kTableBytes) e = hipMalloc(&own, tmp_bytes);
    bool done = false;
    do {
        if (e != hipSuccess) break;
        tmp = own ? own : block + at_table;
        uint2* const raw = reinterpret_cast<uint2*>(tmp);
        uint32_t* const masks = reinterpret_cast<uint32_t*>(tmp + at_masks);
        uint32_t* const words = reinterpret_cast<uint32_t*>(tmp + at_words);
        uint64_t* const sums = reinterpret_cast<uint64_t*>(tmp + at_sums);
        uint4* const base = reinterpret_cast<uint4*>(tmp + at_base);
        uint4* const d_top = reinterpret_cast<uint4*>(tmp + at_top);
        OctFlags* const flags = reinterpret_cast<OctFlags*>(block + at_flags);
        v->root_tag = root_leaf ? (kTagLeaf | ((w[8] & 0xFFFFFFu) || wide ? 0u : kTagEmpty)) : 0u;
        const uint32_t empty_tag = wide ? 0u : kTagEmpty;
        hipLaunchKernelGGL(k_oct_init, dim3((uint32_t)((n + 255 + 256) / 256)), dim3(256), 0, s, masks, words, n, flags);
        if ((e = hipGetLastError()) != hipSuccess ||
            (e = hipMemcpyAsync(raw, w, n * kNodeWords * 4, hipMemcpyHostToDevice, s)) != hipSuccess ||
            (!top.empty() &&
             (e = hipMemcpyAsync(d_top, top.data(), top.size() * sizeof(uint4), hipMemcpyHostToDevice, s)) != hipSuccess))
            break;
        hipLaunchKernelGGL(k_oct_mark_top, dim3(1), dim3(128), 0, s, d_top, (uint32_t)top.size(), masks);
        hipLaunchKernelGGL(k_oct_classify, dim3(blocks), dim3(kOctBlock), 0, s, raw, (uint32_t)n, masks, flags, sums);
        hipLaunchKernelGGL(k_oct_scan, dim3(1), dim3(kOctBlock), 0, s, sums, blocks, base, flags);
        if ((e = hipGetLastError()) != hipSuccess ||
            (e = hipMemcpyAsync(&f, flags, sizeof(f), hipMemcpyDeviceToHost, s)) != hipSuccess ||
            (e = hipStreamSynchronize(s)) != hipSuccess)
            break;
        // every node but the root is a child once: 1 + 8 * internal nodes, none of them twice.
        // The children numbered are as many as the nodes then, and every index k_oct_number
        // and k_oct_emit make is below n, also where a node further down is named twice.
        if (f.refused || 1 + 8ull * f.total[3] != n) break;
        uint64_t numbered = 0;
        for (int q = 0; q < 3; ++q) numbered += (uint64_t)count[q] + f.total[q];
        if (numbered != n) break;
        const uint32_t max_depth = f.total[3] ? f.inner_depth + 1 : 0;
        if (max_depth > 23) break;
        OctBases B;
        for (int q = 0; q < 3; ++q) B.after_top[q] = count[q];
        B.leaf_base = count[0] + f.total[0];
        B.empty_base = B.leaf_base + count[1] + f.total[1];
        const bool depth_bits = !wide && n <= (uint64_t)kRopeIndexMask + 1 && f.depth < 32;
        const uint32_t index_mask = depth_bits ? kRopeIndexMask : wide ? kWideIndexMask : kIndexMask;
        // the records follow the leaves' ropes, in the two words a leaf that six
        // planes leave of the eight the footprint counts
        const uint64_t rec_at = (rope_plane_words(n, B.leaf_base) + 3) & ~3ull;
        if (!root_leaf && rec_at + (uint64_t)kRecWords * B.leaf_base > n * 8) break;
        v->d_cw = reinterpret_cast<uint32_t*>(block);
        v->d_meta = reinterpret_cast<uint32_t*>(block + at_meta);
        v->d_table = reinterpret_cast<uint2*>(block + at_table);
        v->one_block = true;
        uint4* const rec = reinterpret_cast<uint4*>(v->d_cw + rec_at);
        hipLaunchKernelGGL(k_oct_number, dim3(blocks), dim3(kOctBlock), 0, s, raw, (uint32_t)n, masks, base, d_top, B,
                           v->root_tag, empty_tag, depth_bits ? 1u : 0u, words);
        hipLaunchKernelGGL(k_oct_emit, dim3(blocks), dim3(kOctBlock), 0, s, raw, (uint32_t)n, masks, base, d_top, B,
                           empty_tag, index_mask, words, v->d_cw, rec, v->d_meta, flags);
        const bool check_ropes = f.ropes && max_depth >= kRopeCellFirst && max_depth <= kRopeCellLast;
        const auto launch_check_ropes = [&] {
            hipLaunchKernelGGL(k_check_ropes, dim3((uint32_t)(kTableCells / 256)), dim3(256), 0, s, v->d_cw, v->d_meta,
                               (uint32_t)n, B.leaf_base, index_mask, max_depth, v->d_table, flags);
            return hipGetLastError();
        };
        if ((e = hipGetLastError()) != hipSuccess ||
            (e = launch_start_table(v->d_cw, v->root_tag, index_mask, table_shift_of(max_depth), root_leaf ? nullptr : rec, &flags->twice, v->d_table, s)) != hipSuccess ||
            (check_ropes && (e = launch_check_ropes()) != hipSuccess) ||
            (e = hipMemcpyAsync(&f, flags, sizeof(f), hipMemcpyDeviceToHost, s)) != hipSuccess ||
            (e = hipStreamSynchronize(s)) != hipSuccess)
            break;
        if (f.twice) break;
        v->rope_cells = check_ropes && !f.bad_rope;
        v->max_depth = max_depth;
        v->is_rope = f.ropes;
        v->depth_exact = 1;
        v->rope_depth = depth_bits ? 1u : 0u;
        v->index_mask = index_mask;
        v->empty_tag = empty_tag;
        v->empty_start = wide ? B.empty_base : 0xFFFFFFFFu;
        v->leaf_base = B.leaf_base;
        v->rec_at = root_leaf ? 0 : rec_at;
        done = true;
    } while (false);
    if (e != hipSuccess) (void)hipGetLastError();  // reported by the host path if it fails as well
    if (!done || own) (void)hipStreamSynchronize(s);  // nothing may use what is released
    if (own) (void)hipFree(own);
    if (!done) {
        if (block) (void)hipFree(block);
        v->d_cw = v->d_meta = nullptr;
        v->d_table = nullptr;
        v->one_block = false;
        v->root_tag = 0;
    }
    return done;
}

}  // namespace xd
