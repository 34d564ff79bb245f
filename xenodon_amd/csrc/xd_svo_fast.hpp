// Octree traversals on the derived device layout (tagged child words).
//
// Layout: child_w[n*8 + k] = index of child k | kTagLeaf if that child is a
// leaf | kTagEmpty if it is a leaf whose RGB is zero; meta[n] = {color,
// is_leaf_depth}.  A leaf's child words are its ropes, tagged the same way.
// Trees above 2^30 nodes carry 31-bit indices and no empty tag; their empty
// leaves are the indices from a threshold on (empty_mask and empty_min of
// FastSvo cover both).
// Two kinds of walk.  The general ones (fast_df, fast_esvo, fast_rope) take the
// shaders' steps (see xd_svo_ref.hpp) and change only the loads; fast_naive,
// fast_esvo_cells, fast_rope_cells and fast_df_rec take other steps to the same
// leaves, and say why every float that reaches a sum is the shader's.  In both:
//   * "is this node a leaf?" comes with the pointer that led to it, so a
//     descent costs one dependent load per level instead of two;
//   * the colour of an empty leaf is known to be 0 without a load (the sum
//     still adds 0 * step, exactly as the shader does);
//   * svo-df fetches a node's eight child words with two 16-byte loads and
//     then steps through its children from registers.
#pragma once

#include "xd_svo_ref.hpp"
#include "xd_table.hpp"

namespace xd {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct FastSvo {
    const uint32_t* cw;
    const uint32_t* meta;  // colours of nodes [0, n), then their is_leaf_depth words
    uint32_t root_tag;     // kTagLeaf / kTagEmpty of node 0
    const uint32_t* top;   // LDS copy of the child words of nodes [0, n_top)
    uint32_t n_top;
    uint32_t n;            // node count (indices read back from a stack are clamped to it)
    uint32_t depth_exact;  // depth fields of internal nodes equal their tree depth
    const uint2* table;    // start table: kTableCells entries {child word, level}, or null
    uint32_t table_shift;  // ... of cells coarser by this many levels
    uint32_t rope_depth;   // ropes carry their targets' depth fields (kRopeDepthShift)
    uint32_t index_mask;   // index bits of a child word
    // a child word wd names an empty leaf iff (wd & empty_mask) >= empty_min:
    // {kTagEmpty, kTagEmpty} where leaves carry the empty tag, else {index
    // mask, first empty leaf index} (see make_fast_svo)
    uint32_t empty_mask;
    uint32_t empty_min;
    uint32_t leaf_base;    // first leaf: the leaves' ropes are stored as six planes
};

// Rope k of a leaf (its k-th child word): in the plane of rope k for leaves
// from leaf_base on, else (a leaf root) in its own grouped record.
__device__ __forceinline__ uint32_t rope_at(const FastSvo& s, uint32_t leaf, uint32_t k) {
    const uint64_t i = leaf >= s.leaf_base
                           ? (uint64_t)s.leaf_base * 8 + (uint64_t)k * (s.n - s.leaf_base) + (leaf - s.leaf_base)
                           : (uint64_t)leaf * 8 + k;
    return *(const __attribute__((address_space(1))) uint32_t*)(s.cw + i);
}

// The iteration cap as a 32-bit count (a runaway guard that well-formed
// input never reaches; 32-bit counting saves two instructions per step).
__device__ __forceinline__ uint32_t cap32_of(uint64_t cap) { return cap > 0xFFFFFFFFull ? 0xFFFFFFFFu : (uint32_t)cap; }

// A child word names a leaf with zero RGB (whose colour need not be loaded).
__device__ __forceinline__ bool empty_leaf(const FastSvo& s, uint32_t wd) { return (wd & s.empty_mask) >= s.empty_min; }

// FastSvo of a tagged tree.  empty_tag = kTagEmpty marks empty leaves by
// that bit (wd & kTagEmpty is 0 or kTagEmpty, and those layouts set
// empty_start to 0xFFFFFFFF, which no index reaches); empty_tag = 0 by the
// index range from empty_start on.  One comparison covers both.
__device__ __forceinline__ FastSvo make_fast_svo(const uint32_t* cw, const uint32_t* meta, uint32_t root_tag,
                                                 const uint32_t* top, uint32_t n_top, uint32_t n, uint32_t depth_exact,
                                                 const uint2* table, uint32_t table_shift, uint32_t rope_depth, uint32_t index_mask,
                                                 uint32_t empty_tag, uint32_t empty_start, uint32_t leaf_base) {
    return FastSvo{cw, meta, root_tag, top, n_top, n, depth_exact, table, table_shift, rope_depth, index_mask,
                   empty_tag ? empty_tag : index_mask, empty_tag ? empty_tag : empty_start, leaf_base};
}

// Child word k of node n: from LDS for the breadth-first top levels.
__device__ __forceinline__ uint32_t cw_at(const FastSvo& s, uint32_t n, uint32_t k) {
    if (n < s.n_top) return *(const __attribute__((address_space(3))) uint32_t*)(s.top + n * 8 + k);
    return *(const __attribute__((address_space(1))) uint32_t*)(s.cw + (uint64_t)n * 8 + k);
}

// GLSL mod(x, y) for y = 2^k: x / y == x * 2^-k exactly (no rounding in
// either), so the division is a multiplication by the exact reciprocal.
__device__ __forceinline__ float pmod(float x, float y, float inv_y) { return x - y * __builtin_floorf(x * inv_y); }

__device__ __forceinline__ uint32_t colour_if(const FastSvo& s, uint32_t node, uint32_t tag) {
    return empty_leaf(s, tag) ? 0u : s.meta[node];
}

// The child choices of find() at every level, packed: bit (22 - l) of
// level_bits(p) is the comparison p >= offset + extent made at level l.  At
// level l, offset + extent = (2m + 1) * 2^-(l+1) for the integer m that the
// earlier choices fix, and offset is exactly that dyadic value (sums of
// powers of two below 1 are exact in FP32 over the first 23 levels).  For p
// in [0, 1) the comparison is therefore bit 0 of floor(p * 2^(l+1)), which is
// bit (22 - l) of floor(p * 2^23); p < 0 (or NaN) fails every comparison and
// p >= 1 passes every one.
__device__ __forceinline__ uint32_t floor_bits(float p) {
    // the conversion gives 0 for negative numbers and NaN, and the largest word
    // for numbers beyond it
    uint32_t b;
    asm("v_cvt_u32_f32 %0, %1" : "=v"(b) : "v"(p));
    return b;
}
__device__ __forceinline__ uint32_t level_bits(float p) { return min(floor_bits(p * 8388608.0f), (1u << 23) - 1u); }

// x clamped to [lo, hi], one instruction.
__device__ __forceinline__ int32_t clamp3(int32_t x, int32_t lo, int32_t hi) {
    int32_t r;
    asm("v_med3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "v"(lo), "v"(hi));
    return r;
}
__device__ __forceinline__ uint32_t clamp3(uint32_t x, uint32_t lo, uint32_t hi) {
    uint32_t r;
    asm("v_med3_u32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "v"(lo), "v"(hi));
    return r;
}

// The index in s's table.  A branch that all lanes take alike: three shifts by 0 in
// each step of a ray had cost the walks 3 to 4 % on a 9-level tree.
__device__ __forceinline__ uint32_t table_index(const FastSvo& s, uint32_t x, uint32_t y, uint32_t z) {
    uint32_t at;
    if (s.table_shift == 0) {
        at = table_cell(x, y, z);
    } else {
        at = table_cell(x >> s.table_shift, y >> s.table_shift, z >> s.table_shift);
        asm volatile("" : "+v"(at));  // or the compiler makes one computation of the two again
    }
    return at;
}

// svo_naive.comp:8-27 with tagged pointers.  `tag` returns the found node's
// tags.  With a start table the walk begins at the node the table holds for
// the point's level-kTableLevel cell (found from the point's level bits): the same node
// the first kTableLevel levels of the walk reach, with the same offset and extent,
// which are exact dyadic values.
__device__ __forceinline__ uint32_t fast_find(const FastSvo& s, f3 pos, f3& base, float& side, uint32_t& tag) {
    float extent = 1.0f;
    uint32_t index = 0;
    uint32_t level = 0;
    f3 offset = splat(0.0f);
    tag = s.root_tag;
    if (s.table) {
        const uint32_t bx = level_bits(pos.x), by = level_bits(pos.y), bz = level_bits(pos.z);
        const uint2 e = s.table[table_index(s, bx, by, bz)];
        index = e.x & s.index_mask;
        tag = e.x;
        level = e.y & kTableLevelMask;
        extent = __builtin_ldexpf(1.0f, -(int)level);
        const uint32_t c = 23u - level;  // 32-bit shifts: level >= 1 here, or the bits are unused
        offset = level == 0 ? splat(0.0f)
                            : smul(extent, mk((float)(bx >> c), (float)(by >> c), (float)(bz >> c)));
    }
    for (;; ++level) {
        if ((tag & kTagLeaf) || level > kMaxLevels) {
            base = offset;
            side = extent;
            return index;
        }
        extent = extent * 0.5f;
        bool mx = pos.x >= offset.x + extent;
        bool my = pos.y >= offset.y + extent;
        bool mz = pos.z >= offset.z + extent;
        uint32_t child = (mx ? 4u : 0u) + (my ? 2u : 0u) + (mz ? 1u : 0u);
        offset = add(offset, mul(mk(mx ? 1.0f : 0.0f, my ? 1.0f : 0.0f, mz ? 1.0f : 0.0f), splat(extent)));
        const uint32_t wd = cw_at(s, index, child);
        index = wd & s.index_mask;
        tag = wd;
    }
}

// The head of an internal node's record (RenderParams::rec).
struct NodeRec {
    uint32_t inner;  // first internal child
    uint32_t masks;  // bits 0..7: internal children, 8..15: leaves with colour
};

typedef const __attribute__((address_space(1))) uint32_t* GlobalWords;

__device__ __forceinline__ GlobalWords rec_words(const uint4* rec, uint32_t node) {
    return (GlobalWords)rec + (uint64_t)node * kRecWords;
}
__device__ __forceinline__ NodeRec load_rec(GlobalWords w) {
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    const u32x2 v = *(const __attribute__((address_space(1))) u32x2*)w;
    return NodeRec{v.x, v.y};
}

// Computes v here: a sum that the compiler moves down past the load of its next
// term makes the loop wait for that load in the same trip (199x143 frames of a
// 128^3 volume by svo-naive: 0.120 -> 0.104 ms).
__device__ __forceinline__ void pin(f3& v) { asm volatile("" : "+v"(v.x), "+v"(v.y), "+v"(v.z)); }

// The leaf at the position with the bits bx, by, bz, from its cell's table entry:
// its level, and its colour or null for none.  On records a node says of each
// child whether it is a leaf and whether all of its own children are, so the leaf
// is known one load earlier than by child words, and its colour is beside the
// masks: 1080p frames of a 10-level tree (700x490x700 voxels) by svo-naive 1.38 /
// 1.19 / 0.99 -> 1.05 / 0.87 / 0.86 ms.  One address for a leaf of either kind,
// selected, cost 6 % on a 9-level tree.
__device__ __forceinline__ uint32_t table_leaf(const FastSvo& s, const uint4* __restrict__ rec, uint2 e, uint32_t bx,
                                               uint32_t by, uint32_t bz, const uint32_t*& colour) {
    const auto octant = [&](uint32_t level) {
        const uint32_t d = 22u - min(level, 22u);
        return (bx >> d & 1u) << 2 | (by >> d & 1u) << 1 | (bz >> d & 1u);
    };
    const auto colour_in = [&](uint32_t node, uint32_t k) {  // of leaf k; 0 for an empty one
        return reinterpret_cast<const uint32_t*>(rec) + (uint64_t)node * kRecWords + 4u + k;
    };
    uint32_t word = e.x, level = e.y & kTableLevelMask;
    if (e.y & kTableLowNode) {
        colour = colour_in(word & s.index_mask, octant(kTableLevel));
        return kTableLevel + 1;
    }
    if (__builtin_expect(!(word & kTagLeaf), 0)) {
        if (rec) {
            for (;; ++level) {
                const NodeRec r = load_rec(rec_words(rec, word & s.index_mask));
                const uint32_t bit = 1u << octant(level);
                if (!(r.masks & bit)) break;
                word = r.inner + __popc(r.masks & (bit - 1u) & 0xFFu);
                if (r.masks & (bit << 16)) {
                    ++level;
                    break;
                }
            }
            colour = colour_in(word & s.index_mask, octant(level));
            return level + 1;
        }
        for (; !(word & kTagLeaf) && level <= kMaxLevels; ++level) word = cw_at(s, word & s.index_mask, octant(level));
    }
    colour = empty_leaf(s, word) ? nullptr : s.meta + (word & s.index_mask);
    return level;
}

// svo_naive.comp:29-71.  A step's position depends on the box of the leaf before
// it, so a ray is one chain of loads; what is not on it is kept off it:
//  * the start table says where a cell's node has only leaves for children.
//    Such a child's box follows from the position's bits, so the step goes on
//    without waiting for its word;
//  * a leaf's colour is added one step late, while the next step's table entry
//    is on its way;
//  * a step that stays in its cell keeps the entry (rays almost parallel to a
//    plane advance by min_step for thousands of steps).
// Plain 1080p frames of a 512x361x512 volume (outside / over it / inside): 0.70
// / 0.63 / 1.96 -> 0.52 / 0.50 / 1.50 ms, the table in 4x4x4 cells included.
__device__ __forceinline__ f3 fast_naive(const FastSvo& s, const uint4* __restrict__ rec, uint64_t cap, f3 ro, f3 rd) {
    const float min_step = 0.00001f;
    f3 rrd = divv(splat(1.0f), rd);
    f3 bias = mul(rrd, ro);
    f3 box_min = neg(bias);
    f3 box_max = sub(rrd, bias);
    float t_min = max_elem(vmin(box_min, box_max));
    float t_max = min_elem(vmax(box_min, box_max));
    if (t_min > t_max) return splat(0.0f);
    t_min = gmax(t_min, 0.0f);
    f3 total = splat(0.0f);
    float t = t_min + min_step;
    const uint32_t cap32 = cap32_of(cap);
    uint32_t it = 0;
    uint32_t cell = ~0u;
    uint2 e = make_uint2(0, 0);
    uint32_t pend_col = 0;  // the last leaf's term, added at the next step
    float pend_w = 0.0f;
    while (t < t_max) {
        if (++it > cap32) break;
        const f3 pt = add(smul(t, rd), ro);
        const uint32_t bx = level_bits(pt.x), by = level_bits(pt.y), bz = level_bits(pt.z);
        const uint32_t at = table_index(s, bx, by, bz);
        if (at != cell) {
            e = s.table[at];
            cell = at;
        }
        total = add(total, muls(unorm_rgb(pend_col), pend_w));  // +0 the first time
        pin(total);
        const uint32_t* colour;
        const uint32_t level = table_leaf(s, rec, e, bx, by, bz, colour);
        // 1 + the leaf's corner is its leading bits after the point
        const uint32_t keep = ~0u << (23u - level);
        const f3 offset = mk(u2f(0x3F800000u | (bx & keep)) - 1.0f, u2f(0x3F800000u | (by & keep)) - 1.0f,
                             u2f(0x3F800000u | (bz & keep)) - 1.0f);
        const float side = __builtin_ldexpf(1.0f, -(int)level);
        f3 node_min = sub(mul(offset, rrd), bias);
        f3 node_max = sub(mul(add(offset, splat(side)), rrd), bias);
        float u_min = max_elem(vmin(node_min, node_max));
        float u_max = min_elem(vmax(node_min, node_max));
        u_min = gmax(u_min, 0.0f);
        const float step = gmax(u_max - u_min, min_step);
        t = t + step;
        pend_col = colour ? *colour : 0u;
        pend_w = step;
    }
    return add(total, muls(unorm_rgb(pend_col), pend_w));
}

__device__ __forceinline__ uint32_t pick8(const uint4& lo, const uint4& hi, uint32_t ci) {
    const uint32_t a = (ci & 1u) ? lo.y : lo.x, b = (ci & 1u) ? lo.w : lo.z;
    const uint32_t c = (ci & 1u) ? hi.y : hi.x, d = (ci & 1u) ? hi.w : hi.z;
    const uint32_t e = (ci & 2u) ? b : a, f = (ci & 2u) ? d : c;
    return (ci & 4u) ? f : e;
}


__device__ __forceinline__ uint4 to_uint4(u32x4 v) { return make_uint4(v.x, v.y, v.z, v.w); }

__device__ __forceinline__ void load8(const FastSvo& s, uint32_t node, uint4& lo, uint4& hi) {
    // LDS and global loads kept in their own address spaces (a pointer
    // selected between them would become a slower flat load)
    if (node < s.n_top) {
        const __attribute__((address_space(3))) u32x4* p =
            (const __attribute__((address_space(3))) u32x4*)(s.top + node * 8);
        lo = to_uint4(p[0]);
        hi = to_uint4(p[1]);
    } else {
        const __attribute__((address_space(1))) u32x4* p =
            (const __attribute__((address_space(1))) u32x4*)(s.cw + (uint64_t)node * 8);
        lo = to_uint4(p[0]);
        hi = to_uint4(p[1]);
    }
}

// Slab values of the three planes per axis shared by a node's eight child
// boxes: p0 = corner, p1 = corner + side, p2 = p1 + side; T = p * rrd - bias.
// Child box k has, per axis, box_min = T[b] and box_max = T[b + 1] with b the
// axis bit of k -- the same floats svo_df.comp computes from pos and pos+side.
struct Planes {
    float x0, x1, x2, y0, y1, y2, z0, z1, z2;
};

__device__ __forceinline__ Planes node_planes(f3 corner, float side, f3 rrd, f3 bias) {
    Planes P;
    const float px1 = corner.x + side, py1 = corner.y + side, pz1 = corner.z + side;
    P.x0 = corner.x * rrd.x - bias.x;
    P.x1 = px1 * rrd.x - bias.x;
    P.x2 = (px1 + side) * rrd.x - bias.x;
    P.y0 = corner.y * rrd.y - bias.y;
    P.y1 = py1 * rrd.y - bias.y;
    P.y2 = (py1 + side) * rrd.y - bias.y;
    P.z0 = corner.z * rrd.z - bias.z;
    P.z1 = pz1 * rrd.z - bias.z;
    P.z2 = (pz1 + side) * rrd.z - bias.z;
    return P;
}

// t_min / t_max of child box ci of a node: the slab values of node_planes for
// the child's side of each axis (same operations, same floats).
__device__ __forceinline__ void child_trange(f3 corner, float side, f3 rrd, f3 bias, uint32_t ci, float& t_min,
                                             float& t_max) {
    const float px = (ci & 4u) ? corner.x + side : corner.x;
    const float py = (ci & 2u) ? corner.y + side : corner.y;
    const float pz = (ci & 1u) ? corner.z + side : corner.z;
    const float ax = px * rrd.x - bias.x, bx = (px + side) * rrd.x - bias.x;
    const float ay = py * rrd.y - bias.y, by = (py + side) * rrd.y - bias.y;
    const float az = pz * rrd.z - bias.z, bz = (pz + side) * rrd.z - bias.z;
    t_min = max_elem(mk(gmin(ax, bx), gmin(ay, by), gmin(az, bz)));
    t_max = min_elem(mk(gmax(ax, bx), gmax(ay, by), gmax(az, bz)));
}

// Per axis, the near and far plane values of the low ([T0, T1]) and of the high
// ([T1, T2]) children.
struct SlabPairs {
    float xa0, xa1, xb0, xb1, ya0, ya1, yb0, yb1, za0, za1, zb0, zb1;
};

__device__ __forceinline__ SlabPairs slab_pairs(const Planes& P) {
    return SlabPairs{gmin(P.x0, P.x1), gmax(P.x0, P.x1), gmin(P.x1, P.x2), gmax(P.x1, P.x2),
                     gmin(P.y0, P.y1), gmax(P.y0, P.y1), gmin(P.y1, P.y2), gmax(P.y1, P.y2),
                     gmin(P.z0, P.z1), gmax(P.z0, P.z1), gmin(P.z1, P.z2), gmax(P.z1, P.z2)};
}

// Bit k set when child box k of the node is hit (t_min < t_max && t_max > 0,
// svo_df.comp:25-32).  min/max of finite floats are exact, so these are the
// same comparisons as the shader's per-child test.  The two comparisons are
// taken as one, t_max > max(t_min, 0): equal for non-NaN values, and t_min is
// NaN only when all three of its axis minima are, whose axis pairs then give a
// NaN t_max too, so both forms are false there.  The 0 joins the y/z partial
// maxima that the eight children share.
__device__ __forceinline__ void slab_range(const SlabPairs& S, uint32_t k, float& lo, float& hi) {
    const float lo_yz = gmax(gmax((k & 2u) ? S.yb0 : S.ya0, (k & 1u) ? S.zb0 : S.za0), 0.0f);
    lo = gmax((k & 4u) ? S.xb0 : S.xa0, lo_yz);
    hi = gmin((k & 4u) ? S.xb1 : S.xa1, gmin((k & 2u) ? S.yb1 : S.ya1, (k & 1u) ? S.zb1 : S.za1));
}
__device__ __forceinline__ uint32_t slab_hits(const SlabPairs& S) {
    uint32_t m = 0;
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) {
        float lo, hi;
        slab_range(S, k, lo, hi);
        m |= (hi > lo) ? (1u << k) : 0u;
    }
    return m;
}

__device__ __forceinline__ uint32_t child_hits(const Planes& P) { return slab_hits(slab_pairs(P)); }

// svo_df.comp:6-66.  The shader walks the children of a node in index order,
// testing each box, and keeps (node, child index) on a stack.  Here a node's
// eight box tests are done at once into a hit mask, and only hit children are
// visited -- still in index order, so leaves are summed in the shader's order
// with the shader's t values.  A stack entry is (node, children still to
// visit, last visited child, depth); a node with none left is not pushed (the
// shader pops it and finds nothing more to do).  Each iteration visits one hit child and then
// enters at most one node -- the child (descent) or the nearest ancestor with
// children left (pop) -- through one shared path, so lanes that descend and
// lanes that pop wait on the same loads.  The child position the shader
// carries in `pos` is recomputed where it is needed: on descent (corner +
// side on the set axes) and on pop (the shader's pos - mod(pos, 2 * side),
// svo_df.comp:50-61, from a point inside the node being finished, which lies
// inside every ancestor).  The popped node's depth is the depth field the
// shader reads (svo_df.comp:58); when every depth field equals the node's
// depth in the tree, the depth kept on the stack is that same value.  When
// they do not, a popped node can be placed elsewhere than where it was
// entered, so the walk follows the shader literally: every non-last child
// pushes, and a popped node's remaining children are tested again.  EXACT
// selects the first walk (the tree's depth fields are exact, s.depth_exact);
// each walk is built on its own so that neither carries the other's code.
template <bool EXACT>
__device__ __forceinline__ f3 fast_df(const FastSvo& s, uint64_t cap, uint32_t slots, f3 ro, f3 rd,
                                      uint32_t* stk_node, uint32_t* stk_child) {
    f3 rrd = divv(splat(1.0f), rd);
    f3 bias = mul(rrd, ro);
    const int cap_sp = (int)slots;
    int sp = 0;
    uint32_t node = 0, depth = 0;
    f3 corner = splat(0.0f);
    float side = 0.5f;
    f3 total = splat(0.0f);
    uint4 lo, hi;
    load8(s, node, lo, hi);
    uint32_t mask = child_hits(node_planes(corner, side, rrd, bias));
    const uint32_t cap32 = cap32_of(cap);
    uint32_t it = 0;
    for (;;) {
        bool pop = true;
        if (mask != 0) {
            if (++it > cap32) break;
            const uint32_t ci = (uint32_t)__builtin_ctz(mask);
            mask &= mask - 1u;
            bool push;
            const uint32_t wd = pick8(lo, hi, ci);
            const bool bx = (ci & 4u) != 0, by = (ci & 2u) != 0, bz = (ci & 1u) != 0;
            if (wd & kTagLeaf) {
                if (!empty_leaf(s, wd)) {  // an empty leaf adds exactly +0
                    float t_min, t_max;
                    child_trange(corner, side, rrd, bias, ci, t_min, t_max);
                    total = add(total, muls(unorm_rgb(s.meta[wd & s.index_mask]), t_max - gmax(t_min, 0.0f)));
                }
                if (mask != 0) continue;  // next sibling, from registers
            } else if (!(push = EXACT ? mask != 0 : ci != 7u) || sp < cap_sp) {
                if (push) {
                    stk_node[sp * kWaveLanes] = node;
                    stk_child[sp * kWaveLanes] = mask | (ci << 8) | (depth << 11);
                    ++sp;
                }
                corner = mk(bx ? corner.x + side : corner.x, by ? corner.y + side : corner.y,
                            bz ? corner.z + side : corner.z);
                side = side * 0.5f;
                node = wd & s.index_mask;
                depth = depth + 1u;
                pop = false;
            } else if (mask != 0) {
                continue;  // stack full: the shader skips this child
            }
        }
        if (pop) {
            if (sp == 0) break;
            --sp;
            node = min(stk_node[sp * kWaveLanes], s.n - 1u);
            const uint32_t e = stk_child[sp * kWaveLanes];
            mask = e & 0xFFu;
            depth = (e >> 11) & 0xFFu;
            const uint32_t d = EXACT ? depth : (s.meta[(uint64_t)s.n + node] & kDepthMask);
            const f3 pos = mk(corner.x + side, corner.y + side, corner.z + side);
            side = __builtin_ldexpf(1.0f, -(int)d) * 0.5f;
            if (EXACT) {
                // The tree's geometry: pos and every corner are multiples of
                // 2^-23 in [0, 1] (at most 23 levels), and s2 = 2^-d.  Then
                // pos * 2^d, its floor times s2 and both subtractions of
                // pos - mod(pos, s2) are exact, so that corner is the
                // product s2 * floor(pos * 2^d).
                const float s2 = side * 2.0f, inv = __builtin_ldexpf(1.0f, (int)d);
                corner = mk(s2 * __builtin_floorf(pos.x * inv), s2 * __builtin_floorf(pos.y * inv),
                            s2 * __builtin_floorf(pos.z * inv));
            } else {
                // side is a power of two, so mod(pos, 2 side) is exact with the reciprocal
                const float s2 = side * 2.0f;
                const float inv = __builtin_ldexpf(1.0f, -__builtin_amdgcn_frexp_expf(s2) + 1);
                corner = sub(pos, mk(pmod(pos.x, s2, inv), pmod(pos.y, s2, inv), pmod(pos.z, s2, inv)));
            }
        }
        load8(s, node, lo, hi);
        if (!pop) {
            mask = child_hits(node_planes(corner, side, rrd, bias));
        } else if (!EXACT) {
            // the shader tests the remaining children at the geometry the
            // depth field gives the popped node, which may differ from the
            // geometry they were first tested at
            const uint32_t ci = (stk_child[sp * kWaveLanes] >> 8) & 7u;
            mask = child_hits(node_planes(corner, side, rrd, bias)) & (0xFEu << ci) & 0xFFu;
        }
    }
    return total;
}

// The children that a ray passes in a node, in its order, and for how long.
//
// A line passes at most four of the eight: the near one first, then across the
// middle planes in the order of their t.  With E the last near plane (0 at least),
// X the first far plane and s1 <= s2 <= s3 the middle planes, child j's t-range is
// [max(E, s_j), min(X, s_j+1)].  These are the floats of the box test, the greatest
// near and the least far plane of the child's own six, since along each axis near
// <= middle <= far after rounding as well; a child that crosses the planes in
// another order has no length.  Of two equal middle planes either comes first: the
// child between them has none.  All planes must be finite (df_ray).
struct Passed {
    float whole;            // of the node itself
    float length[4];        // above 0 for a child that the box test hits
    uint32_t axis1, axis3;  // index bits of the first and the last middle plane's axis
};
__device__ __forceinline__ Passed passed_children(const Planes& P) {
    const float e = gmax(max_elem(mk(gmin(P.x0, P.x2), gmin(P.y0, P.y2), gmin(P.z0, P.z2))), 0.0f);
    const float x = min_elem(mk(gmax(P.x0, P.x2), gmax(P.y0, P.y2), gmax(P.z0, P.z2)));
    const f3 m = mk(P.x1, P.y1, P.z1);
    const float s1 = min_elem(m), s2 = __builtin_amdgcn_fmed3f(m.x, m.y, m.z), s3 = max_elem(m);
    Passed c;
    c.whole = x - e;
    c.length[0] = gmin(x, s1) - e;
    c.length[1] = gmin(x, s2) - gmax(e, s1);
    c.length[2] = gmin(x, s3) - gmax(e, s2);
    c.length[3] = x - gmax(e, s3);
    c.axis1 = m.x == s1 ? 4u : m.y == s1 ? 2u : 1u;
    c.axis3 = m.x == s3 ? 4u : m.y == s3 ? 2u : 1u;
    return c;
}

__device__ __forceinline__ bool df_ray(f3 rrd, f3 bias) {
    return fabs_(bias.x) <= 1e30f && fabs_(bias.y) <= 1e30f && fabs_(bias.z) <= 1e30f && fabs_(rrd.x) <= 1e30f &&
           fabs_(rrd.y) <= 1e30f && fabs_(rrd.z) <= 1e30f;
}

// The smaller key first.
__device__ __forceinline__ void order(uint32_t& ka, float& a, uint32_t& kb, float& b) {
    const bool swap = kb < ka;
    const float f = swap ? b : a;
    b = swap ? a : b;
    a = f;
    const uint32_t k = min(ka, kb);
    kb = max(ka, kb);
    ka = k;
}

// The walk of fast_df<true> on records, for rays that df_ray accepts.  It is bound
// by the instructions it issues, half of the lanes busy, so it is built to need
// fewer:
//  * empty leaves, which add exactly +0, leave the hit mask at once;
//  * a trip takes one child, whatever it is: the planes of its box are a leaf's
//    t-range, an internal node's hit test and the t-ranges of its children;
//  * a node without internal children -- most of the leaves with colour are under
//    such -- is summed from its parent, the four children that the ray passes in
//    index order, so it costs no push and no pop;
//  * a node that is finished is popped, and the ancestor's next child taken, in the
//    same trip.
// Plain 1080p frames of a 512x361x512 volume 1.22 / 1.40 / 4.20 -> 0.98 / 1.13 /
// 3.33 ms, the three batched 6.12 -> 4.93, a 199x143 frame of a 128^3 volume 0.171
// -> 0.138, against eight box tests a node and a sum in child order with each of the
// eight under a condition.  Entering the nodes without internal children took 1.05 /
// 1.18 / 3.43, and the head's load after the planes 1.05 / 1.14 / 3.39.
__device__ __forceinline__ f3 fast_df_rec(const uint4* __restrict__ rec, uint32_t n, uint64_t cap, f3 rrd, f3 bias,
                                          uint32_t* stk_node, uint32_t* stk_child) {
    int sp = 0;  // at most the tree's depth, below the stack's slots: each ancestor is on it once
    f3 total = splat(0.0f);
    const uint32_t near = (rrd.x < 0.0f ? 4u : 0u) | (rrd.y < 0.0f ? 2u : 0u) | (rrd.z < 0.0f ? 1u : 0u), far = near ^ 7u;
    const uint32_t cap32 = cap32_of(cap);
    uint32_t it = 0;
    // the root as the only child of a node around it
    uint32_t node = 0, depth = ~0u, mask = 1;
    f3 corner = splat(0.0f);
    float side = 1.0f;  // of the node's children
    NodeRec r = NodeRec{0u, (load_rec(rec_words(rec, 0)).masks & 0xFFu) ? 1u : 0x10001u};
    for (;;) {
        if (mask == 0) {
            if (sp == 0) break;
            --sp;
            node = min(stk_node[sp * kWaveLanes], n - 1u);
            const uint32_t e = stk_child[sp * kWaveLanes];
            mask = e & 0xFFu;
            depth = e >> 8;
            side = __builtin_ldexpf(0.5f, -(int)depth);
            // The corner of the ancestor of this depth: every corner is a
            // multiple of 2^-23 below 1, so 1 + corner is exact and its top
            // `depth` fraction bits are the ancestor's.
            const uint32_t keep = ~0u << (23u - depth);
            corner = mk(u2f(f2u(corner.x + 1.0f) & keep) - 1.0f, u2f(f2u(corner.y + 1.0f) & keep) - 1.0f,
                        u2f(f2u(corner.z + 1.0f) & keep) - 1.0f);
            r = load_rec(rec_words(rec, node));
        }
        if (++it > cap32) break;
        const uint32_t rest = mask & (mask - 1u), bit = mask ^ rest;
        mask = rest;
        const bool leaf = (r.masks & (bit << 8)) != 0;
        const uint32_t child = leaf ? node : r.inner + __popc(r.masks & (bit - 1u) & 0xFFu);
        const GlobalWords w = rec_words(rec, child);
        NodeRec next = load_rec(w);  // in flight during the planes' arithmetic; wanted by an internal node
        const f3 at = mk((bit & 0xF0u) ? corner.x + side : corner.x, (bit & 0xCCu) ? corner.y + side : corner.y,
                         (bit & 0xAAu) ? corner.z + side : corner.z);
        Passed c = passed_children(node_planes(at, side * 0.5f, rrd, bias));
        asm volatile(""
                     : "+v"(next.inner), "+v"(next.masks), "+v"(c.length[0]), "+v"(c.length[1]), "+v"(c.length[2]),
                       "+v"(c.length[3]));
        if (leaf) {
            total = add(total, muls(unorm_rgb(w[4 + __builtin_ctz(bit)]), c.whole));
        } else if (r.masks & (bit << 16)) {
            uint32_t k0 = near, k1 = near ^ c.axis1, k2 = far ^ c.axis3, k3 = far;
            order(k0, c.length[0], k1, c.length[1]);
            order(k2, c.length[2], k3, c.length[3]);
            order(k0, c.length[0], k2, c.length[2]);
            order(k1, c.length[1], k3, c.length[3]);
            order(k1, c.length[1], k2, c.length[2]);
            // 0 for empty leaves; a child not passed adds +0
            const uint32_t col[4] = {w[4 + k0], w[4 + k1], w[4 + k2], w[4 + k3]};
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) total = add(total, muls(unorm_rgb(col[j]), gmax(c.length[j], 0.0f)));
        } else {
            if (rest != 0) {
                stk_node[sp * kWaveLanes] = node;
                stk_child[sp * kWaveLanes] = rest | (depth << 8);
                ++sp;
            }
            r = next;
            node = child;
            corner = at;
            side = side * 0.5f;
            depth = depth + 1u;
            mask = (c.length[0] > 0.0f ? 1u << near : 0u) | (c.length[1] > 0.0f ? 1u << (near ^ c.axis1) : 0u) |
                   (c.length[2] > 0.0f ? 1u << (far ^ c.axis3) : 0u) | (c.length[3] > 0.0f ? 1u << far : 0u);
            mask &= (r.masks | (r.masks >> 8)) & 0xFFu;
        }
        // One way back to the top: else the compiler makes a loop of its own of the
        // ways that leave the node as it is, and the lanes in it keep the others waiting
        // (1.35 / 1.71 / 4.32 ms).
        pin(corner);
        asm volatile("" : "+v"(mask), "+v"(node), "+v"(side));
    }
    return total;
}

// svo_rope.comp:65-135 (find_relative inlined).  With s.rope_depth the depth
// field of a rope's target comes with the rope word, so a hop needs no load
// of the target's {color, depth} before its walk; the found leaf's colour is
// loaded together with the next rope.
__device__ __forceinline__ f3 fast_rope(const FastSvo& s, uint64_t cap, f3 ro, f3 rd) {
    f3 sgn = mk(fsign(rd.x), fsign(rd.y), fsign(rd.z));
    const uint32_t nbx = 1u - (sgn.x > 0.0f ? 1u : 0u);
    const uint32_t nby = 3u - (sgn.y > 0.0f ? 1u : 0u);
    const uint32_t nbz = 5u - (sgn.z > 0.0f ? 1u : 0u);
    sgn = add(sgn, splat(0.1f));
    f3 rrd = divv(splat(1.0f), rd);
    f3 bias = mul(rrd, ro);
    f3 box_min = neg(bias);
    f3 box_max = sub(rrd, bias);
    float t_min = max_elem(vmin(box_min, box_max));
    float t_max = min_elem(vmax(box_min, box_max));
    if (t_min > t_max) return splat(0.0f);
    t_min = gmax(t_min, 0.0f);
    const uint32_t rope_mask = s.index_mask;  // kRopeIndexMask when ropes carry depths
    f3 pos = add(ro, smul(t_min, rd));
    f3 offset;
    float side;
    uint32_t tag;
    uint32_t node = fast_find(s, pos, offset, side, tag);
    f3 node_min = sub(mul(offset, rrd), bias);
    f3 node_max = sub(mul(add(offset, splat(side)), rrd), bias);
    f3 far = vmax(node_min, node_max);
    float u_min = max_elem(vmin(node_min, node_max));
    float u_max = min_elem(far);
    float step = u_max - gmax(u_min, 0.0f);
    f3 total = muls(unorm_rgb(colour_if(s, node, tag)), step);
    f3 mask;
    uint32_t n = neighbor_index(nbx, nby, nbz, far, mask);
    uint32_t wd = rope_at(s, node, n);
    node = wd & rope_mask;
    tag = wd;
    offset = add(offset, muls(mul(mask, sgn), side));
    const uint32_t cap32 = cap32_of(cap);
    uint32_t it = 0;
    while (node != 0) {
        if (++it > cap32) break;
        pos = add(ro, smul(u_max, rd));
        // find_relative (svo_rope.comp:29-48) from the rope's target
        const uint32_t start = node;
        uint32_t start_col = 0;
        int d;
        if (s.rope_depth) {
            d = (int)((wd >> kRopeDepthShift) & 31u);
        } else {
            d = (int)(s.meta[(uint64_t)s.n + node] & kDepthMask);
            start_col = s.meta[node];
        }
        float extent = __builtin_ldexpf(1.0f, -d);
        const float inv = __builtin_ldexpf(1.0f, d);
        offset = sub(offset, mk(pmod(offset.x, extent, inv), pmod(offset.y, extent, inv), pmod(offset.z, extent, inv)));
        for (uint32_t level = 0;; ++level) {
            if ((tag & kTagLeaf) || level > kMaxLevels) break;
            extent = extent * 0.5f;
            bool mx = pos.x >= offset.x + extent;
            bool my = pos.y >= offset.y + extent;
            bool mz = pos.z >= offset.z + extent;
            uint32_t child = (mx ? 4u : 0u) + (my ? 2u : 0u) + (mz ? 1u : 0u);
            offset = add(offset, mul(mk(mx ? 1.0f : 0.0f, my ? 1.0f : 0.0f, mz ? 1.0f : 0.0f), splat(extent)));
            wd = cw_at(s, node, child);
            node = wd & s.index_mask;
            tag = wd;
        }
        side = extent;
        node_min = sub(mul(offset, rrd), bias);
        node_max = sub(mul(add(offset, splat(side)), rrd), bias);
        far = vmax(node_min, node_max);
        u_min = max_elem(vmin(node_min, node_max));
        u_max = min_elem(far);
        step = u_max - gmax(u_min, 0.0f);
        const uint32_t col =
            empty_leaf(s, tag) ? 0u : (node == start && !s.rope_depth ? start_col : s.meta[node]);
        n = neighbor_index(nbx, nby, nbz, far, mask);
        wd = rope_at(s, node, n);  // in flight together with the colour
        total = add(total, muls(unorm_rgb(col), step));
        node = wd & rope_mask;
        tag = wd;
        offset = add(offset, muls(mul(mask, sgn), side));
    }
    return total;
}

// The walk of fast_rope for trees whose ropes are those of their geometry
// (k_check_ropes), for rays that rope_cell_ray accepts: a rope leads to the node beside the leaf,
// along the axis of its exit, at the leaf's level or above, and the descent from
// there follows the position.  The leaf is thus the one at the position, clamped to
// the neighbouring cell of the leaf's size: one load of the start table instead of
// the rope and a load a level.  Plain 1080p frames of a 512x361x512 volume 0.66 /
// 0.70 / 1.61 -> 0.49 / 0.56 / 1.67 ms, batched 2.70 -> 2.45; 700x490x700 voxels (10
// levels) 1.92 / 1.85 / 0.99 -> 1.04 / 0.83 / 1.00, batched 4.39 -> 1.66; eight
// frames of shells in 512^3 voxels 53.9 -> 15.7.  fill_params has the rule.
__device__ __forceinline__ bool rope_cell_ray(f3 ro, f3 rd) {  // finite, and times 2^23 as well
    return fabs_(ro.x) <= 1e20f && fabs_(ro.y) <= 1e20f && fabs_(ro.z) <= 1e20f && fabs_(rd.x) <= 2.0f &&
           fabs_(rd.y) <= 2.0f && fabs_(rd.z) <= 2.0f;
}
__device__ __forceinline__ f3 fast_rope_cells(const FastSvo& s, const uint4* __restrict__ rec, uint64_t cap, f3 ro,
                                              f3 rd) {
    f3 rrd = divv(splat(1.0f), rd);
    f3 bias = mul(rrd, ro);
    f3 box_min = neg(bias);
    f3 box_max = sub(rrd, bias);
    float t_min = max_elem(vmin(box_min, box_max));
    float t_max = min_elem(vmax(box_min, box_max));
    if (t_min > t_max) return splat(0.0f);
    float u = gmax(t_min, 0.0f);  // where the ray enters the leaf
    // positions times 2^23, rounded as they are
    const f3 ro23 = muls(ro, 0x1p23f), rd23 = muls(rd, 0x1p23f);
    // the cell that the leaf is in: its lower corner and its low bits
    uint32_t nx = 0, ny = 0, nz = 0, rest = (1u << 23) - 1u;
    f3 total = splat(0.0f);
    uint32_t pend_col = 0;  // the last leaf's term, added at the next step
    float pend_w = 0.0f;
    const uint32_t cap32 = cap32_of(cap);
    uint32_t it = 0;
    do {
        const f3 pos = add(ro23, smul(u, rd23));
        const uint32_t bx = clamp3(floor_bits(pos.x), nx, nx | rest);
        const uint32_t by = clamp3(floor_bits(pos.y), ny, ny | rest);
        const uint32_t bz = clamp3(floor_bits(pos.z), nz, nz | rest);
        const uint2 e = s.table[table_index(s, bx, by, bz)];
        total = add(total, muls(unorm_rgb(pend_col), pend_w));  // +0 the first time
        pin(total);
        const uint32_t* colour;
        const uint32_t level = table_leaf(s, rec, e, bx, by, bz, colour);
        const uint32_t size = 1u << (23u - level), keep = 0u - size;  // keep: the mask, and -size
        // 1 + the leaf's corner is its leading bits after the point
        const f3 offset = mk(u2f(0x3F800000u | (bx & keep)) - 1.0f, u2f(0x3F800000u | (by & keep)) - 1.0f,
                             u2f(0x3F800000u | (bz & keep)) - 1.0f);
        const float side = __builtin_ldexpf(1.0f, -(int)level);
        f3 node_min = sub(mul(offset, rrd), bias);
        f3 node_max = sub(mul(add(offset, splat(side)), rrd), bias);
        f3 far = vmax(node_min, node_max);
        const float u_min = max_elem(vmin(node_min, node_max));
        u = min_elem(far);
        pend_col = colour ? *colour : 0u;
        pend_w = u - gmax(u_min, 0.0f);
        // one past the leaf on the axis of neighbor_index
        rest = size - 1u;
        const bool ax = far.x < gmin(far.y, far.z), ay = far.y < far.z && !ax, az = !ax && !ay;
        nx = (bx & keep) + (ax ? (rd.x > 0.0f ? size : keep) : 0u);
        ny = (by & keep) + (ay ? (rd.y > 0.0f ? size : keep) : 0u);
        nz = (bz & keep) + (az ? (rd.z > 0.0f ? size : keep) : 0u);
        if ((nx | ny | nz) >> 23) break;
    } while (it++ < cap32);
    return add(total, muls(unorm_rgb(pend_col), pend_w));
}

// esvo.comp:30-136, for the trees and rays that fast_esvo_cells does not take.
__device__ __forceinline__ f3 fast_esvo(const FastSvo& s, uint64_t cap, uint32_t slots, f3 ro, f3 rd,
                                        uint32_t* stk_parent, float* stk_tmax) {
    EsvoRay r = esvo_setup(ro, rd);
    float t_min = r.t_min, t_max = r.t_max, h = r.h;
    f3 pos = r.pos;
    uint32_t idx = r.idx, parent = 0, scale = 22;
    float scale_exp2 = 0.5f;
    f3 total = splat(0.0f);
    uint32_t pend_col = 0;  // the last leaf's term, added at the next leaf so that
    float pend_w = 0.0f;    // its colour load overlaps the walk in between
    const uint32_t cap32 = cap32_of(cap);
    uint32_t it = 0;
    while (scale < 23u) {
        if (++it > cap32) break;
        f3 t_corner = sub(mul(pos, r.t_coeff), r.t_bias);
        float tc_max = min_elem(t_corner);
        if (t_min <= t_max) {
            float tv_max = gmin(t_max, tc_max);
            if (t_min <= tv_max) {
                const uint32_t wd = cw_at(s, parent, idx ^ r.octant_mask);
                const uint32_t child = wd & s.index_mask;
                if (wd & kTagLeaf) {
                    const uint32_t col = colour_if(s, child, wd);
                    total = add(total, muls(unorm_rgb(pend_col), pend_w));  // +0 the first time
                    pend_col = col;
                    pend_w = tv_max - t_min;
                } else {
                    if (tc_max < h) {
                        uint32_t slot = 22u - scale;
                        if (slot < slots) {
                            stk_parent[slot * kWaveLanes] = parent;
                            stk_tmax[slot * kWaveLanes] = t_max;
                        }
                    }
                    h = tc_max;
                    parent = child;
                    --scale;
                    scale_exp2 = scale_exp2 * 0.5f;
                    f3 t_center = add(smul(scale_exp2, r.t_coeff), t_corner);
                    bool ax = t_center.x > t_min, ay = t_center.y > t_min, az = t_center.z > t_min;
                    idx = cxor(0u, ax, ay, az);
                    pos = add(pos, mk(ax ? scale_exp2 : 0.0f, ay ? scale_exp2 : 0.0f, az ? scale_exp2 : 0.0f));
                    t_max = tv_max;
                    continue;
                }
            }
        }
        bool ax = t_corner.x <= tc_max, ay = t_corner.y <= tc_max, az = t_corner.z <= tc_max;
        uint32_t step_mask = cxor(0u, ax, ay, az);
        pos = sub(pos, mk(ax ? scale_exp2 : 0.0f, ay ? scale_exp2 : 0.0f, az ? scale_exp2 : 0.0f));
        t_min = tc_max;
        idx ^= step_mask;
        if ((idx & step_mask) != 0) {
            if (!esvo_pop(pos, scale_exp2, scale, idx, ax, ay, az)) break;
            uint32_t slot = 22u - scale;
            parent = slot < slots ? min(stk_parent[slot * kWaveLanes], s.n - 1u) : 0u;
            t_max = slot < slots ? stk_tmax[slot * kWaveLanes] : 0.0f;
            h = 0.0f;
        }
    }
    return add(total, muls(unorm_rgb(pend_col), pend_w));
}

// The walk of fast_esvo from cell to cell, for trees of 1 to kEsvoCellLevels
// levels and rays that esvo_cell_ray accepts.
//
// The shader descends, steps and pops a level a trip; a wave's lanes do these in
// turn, each trip costing what all of them cost.  Here a trip is one leaf, found
// with one load of the start table, and there is no stack.  The terms, their order
// and every float that enters a comparison or a sum are the shader's:
//  * positions are 23-bit numbers, 1 + n * 2^-23 on the mirrored axes.  A descent's
//    choices along an axis, t_center > t_min at each level, depend on that axis
//    alone, and planes far from the ray's position at t_min fall as their distance
//    says.  One plane can be near: the multiple m of the tree's finest cell that is
//    nearest to (t_min + t_bias) * -|rd|.  Its comparison is made, as the shader
//    makes it; the bits below are then 0...0 or 1...1.  (Positions are off by less
//    than 2^-18 here, half of a finest cell is at least 2^-15.)  The descent starts
//    in the cell that the step or pop leads to, so the result is clamped to that.
//  * t_max is the least of the root's and the exits of the nodes entered, and an
//    exit never lies behind its parent's: min(t_max of the root, the leaf's exit).
//  * a node that t_min has passed already (t_center and its plane's t round apart)
//    is skipped whole, so a skipped leaf looks for the outermost such node.
// Plain 1080p frames of the 9-level tree above 1.06 / 1.12 / 3.50 -> 0.65 / 0.69 /
// 2.08 ms, the three batched 4.98 -> 3.15; 10 levels 1.67 / 1.33 / 1.50 -> 1.02
// / 0.82 / 1.09; a DAG without records 1.47 / 1.87 / 2.49 -> 0.86 / 1.08 / 1.51; a
// 199x143 frame of a 128^3 volume 0.178 -> 0.113.
constexpr uint32_t kEsvoCellLevels = 14;

__device__ __forceinline__ bool esvo_cell_ray(f3 ro, f3 rd, const EsvoRay& r) {
    const f3 d = mk(ro.x - 1.5f, ro.y - 1.5f, ro.z - 1.5f);
    return r.t_min <= r.t_max && fabs_(d.x) <= 3.5f && fabs_(d.y) <= 3.5f && fabs_(d.z) <= 3.5f &&
           fabs_(rd.x) <= 2.0f && fabs_(rd.y) <= 2.0f && fabs_(rd.z) <= 2.0f;
}

__device__ __forceinline__ float esvo_plane(int32_t n, float t_coeff, float t_bias) {
    return u2f(0x3F800000u | (uint32_t)n) * t_coeff - t_bias;
}

// The cell along one axis at t_min, within the region of low bits `rest` around n.
struct EsvoSnap {
    float add;      // rounds a position to a multiple of the finest cell
    uint32_t shift, base;
};
__device__ __forceinline__ int32_t esvo_cell(const EsvoSnap& q, float t_min, float neg_rd, float t_coeff, float t_bias,
                                             int32_t n, int32_t rest) {
    const float p = (t_min + t_bias) * neg_rd;
    const int32_t m = (int32_t)((f2u(p + q.add) << q.shift) + q.base);
    const int32_t half = m & -m;  // of the node that plane m divides
    const float t_center = __builtin_fmaf((float)half, t_coeff * 0x1p-23f, esvo_plane(m - half, t_coeff, t_bias));
    return clamp3(t_center > t_min ? m : m - 1, n & ~rest, n | rest);
}

__device__ __forceinline__ f3 fast_esvo_cells(const FastSvo& s, const uint4* __restrict__ rec, uint32_t depth,
                                              uint64_t cap, f3 rd, const EsvoRay& r) {
    const uint32_t levels = max(depth, kTableLevel);
    EsvoSnap q;
    q.shift = 23u - levels;
    q.add = __builtin_ldexpf(1.5f, (int)q.shift);  // its last place is 2^-levels
    q.base = 0u - (f2u(q.add) << q.shift) - (1u << 23);
    const f3 nd = mk(-fabs_(rd.x), -fabs_(rd.y), -fabs_(rd.z));
    const uint32_t fx = (r.octant_mask & 4u) ? 0x7FFFFFu : 0u, fy = (r.octant_mask & 2u) ? 0x7FFFFFu : 0u,
                   fz = (r.octant_mask & 1u) ? 0x7FFFFFu : 0u;
    // the first cell: the root's child that esvo_setup chose
    int32_t nx = (r.idx & 4u) ? 1 << 22 : 0, ny = (r.idx & 2u) ? 1 << 22 : 0, nz = (r.idx & 1u) ? 1 << 22 : 0;
    int32_t rest = (1 << 22) - 1;
    float t_min = r.t_min;
    f3 total = splat(0.0f);
    uint32_t pend_col = 0;  // the last leaf's term, added at the next step
    float pend_w = 0.0f;
    const uint32_t cap32 = cap32_of(cap);
    uint32_t it = 0;
    while (++it <= cap32) {
        const int32_t cx = esvo_cell(q, t_min, nd.x, r.t_coeff.x, r.t_bias.x, nx, rest);
        const int32_t cy = esvo_cell(q, t_min, nd.y, r.t_coeff.y, r.t_bias.y, ny, rest);
        const int32_t cz = esvo_cell(q, t_min, nd.z, r.t_coeff.z, r.t_bias.z, nz, rest);
        const uint32_t bx = (uint32_t)cx ^ fx, by = (uint32_t)cy ^ fy, bz = (uint32_t)cz ^ fz;
        const uint2 e = s.table[table_index(s, bx, by, bz)];
        total = add(total, muls(unorm_rgb(pend_col), pend_w));  // +0 the first time
        pin(total);
        const uint32_t* colour;
        const uint32_t level = table_leaf(s, rec, e, bx, by, bz, colour);
        int32_t size = 1 << (23u - level);
        int32_t lx = cx & -size, ly = cy & -size, lz = cz & -size;
        f3 t_corner = mk(esvo_plane(lx, r.t_coeff.x, r.t_bias.x), esvo_plane(ly, r.t_coeff.y, r.t_bias.y),
                         esvo_plane(lz, r.t_coeff.z, r.t_bias.z));
        float tc_max = min_elem(t_corner);
        const float tv_max = gmin(r.t_max, tc_max);
        pend_col = 0;
        if (t_min <= tv_max) {
            if (colour) pend_col = *colour;
            pend_w = tv_max - t_min;
        } else {
            for (int32_t outer = rest + 1; outer > size; outer >>= 1) {
                const f3 tc = mk(esvo_plane(cx & -outer, r.t_coeff.x, r.t_bias.x),
                                 esvo_plane(cy & -outer, r.t_coeff.y, r.t_bias.y),
                                 esvo_plane(cz & -outer, r.t_coeff.z, r.t_bias.z));
                if (t_min <= gmin(r.t_max, min_elem(tc))) continue;
                size = outer;
                lx = cx & -size;
                ly = cy & -size;
                lz = cz & -size;
                t_corner = tc;
                tc_max = min_elem(tc);
                break;
            }
        }
        nx = lx - (t_corner.x <= tc_max ? size : 0);
        ny = ly - (t_corner.y <= tc_max ? size : 0);
        nz = lz - (t_corner.z <= tc_max ? size : 0);
        if ((nx | ny | nz) < 0) break;
        // the highest bit that changed is the size of the cell that the step leads to
        rest = (int32_t)(0x7FFFFFFFu >> __builtin_clz((uint32_t)((lx ^ nx) | (ly ^ ny) | (lz ^ nz))));
        t_min = tc_max;
    }
    return add(total, muls(unorm_rgb(pend_col), pend_w));
}

}  // namespace xd
