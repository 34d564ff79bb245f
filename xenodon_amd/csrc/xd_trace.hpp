// Per-ray traversal device code shared by the plain kernels (one launch
// per output) and the persistent batch kernel (xd_batch.hip).
#pragma once

#include "xd_internal.hpp"
#include "xd_svo_fast.hpp"

namespace xd {

// Pixel of this lane.  WPB = 4: a block is a 2x2 arrangement of wavefront
// tiles; WPB = 1: a block is one tile.  The 8 XCDs receive blocks
// round-robin (block b runs on XCD b % 8).  chunks = 0 keeps that order, so
// neighbouring blocks run on different XCDs; chunks = N >= 1 cuts the image's
// blocks (row-major) into 8N runs and gives XCD x runs x, x + 8, ..., so each
// XCD's L2 holds the volume behind a few bands while every XCD still gets a
// share of each part of the image (N = 1: one contiguous band per XCD).
template <int TW, int WPB>
__device__ __forceinline__ void block_pixel(uint32_t W, uint32_t H, uint32_t chunks, uint32_t& ix, uint32_t& iy) {
    constexpr uint32_t TH = 64 / TW;
    constexpr uint32_t BW = (WPB == 4 ? 2 : 1) * TW, BH = (WPB == 4 ? 2 : 1) * TH;
    const uint32_t nbx = (W + BW - 1) / BW;
    const uint32_t nblocks = nbx * ((H + BH - 1) / BH);
    const uint32_t b = blockIdx.x;
    uint32_t lb = b;
    if (chunks != 0) {
        const uint32_t run = nblocks / (8u * chunks);  // blocks per run
        if (run != 0 && b < run * 8u * chunks) {
            const uint32_t j = b >> 3;  // j-th block this XCD receives
            lb = ((j / run) * 8u + (b & 7u)) * run + j % run;
        }
    }
    const uint32_t bx = lb % nbx, by = lb / nbx;
    const uint32_t w = threadIdx.x >> 6, lane = threadIdx.x & 63u;
    ix = bx * BW + (WPB == 4 ? (w & 1u) * TW : 0u) + (lane % TW);
    iy = by * BH + (WPB == 4 ? (w >> 1) * TH : 0u) + (lane / TW);
}

__device__ __forceinline__ void add_words(unsigned long long* counter, uint64_t w) {
    // wave-wide sum, one atomic per wavefront
    for (int off = 32; off > 0; off >>= 1) w += __shfl_xor(w, off, 64);
    if ((threadIdx.x & 63u) == 0 && w) atomicAdd(counter, (unsigned long long)w);
}

// GLSL ivec3(vec3) truncation; out-of-range saturates and NaN gives 0.
__device__ __forceinline__ int32_t f2i_sat(float x) {
    if (!(x == x)) return 0;
    if (x >= 2147483647.0f) return 2147483647;
    if (x <= -2147483648.0f) return (-2147483647 - 1);
    return (int32_t)x;
}

// ---------------------------------------------------------------------------
// DDA: resources/dda.comp:13-53
//
// The step sequence (side_dist additions, masks, t) is the shader's, one
// rounding per operation, and so is the order of the sum.  The loop is bound by
// the instructions it issues (0.33 of them a cycle on each SIMD, all lanes
// busy, memory pipes under half busy), so it is built to need few:
//  * steps come in batches of RUN, and a batch looks at the macro mask once.  A
//    mask bit covers its cell and 8 voxels around it, so a clear bit says that
//    none of the batch's texels has colour: each would add exactly +0.  Where
//    it is set, the batch gathers its texels together, without a look at the
//    mask for each.  A look per step had cost as much as the step: plain 1080p
//    frames of a 512x361x512 volume went from 0.76 / 0.84 / 2.00 ms (outside /
//    over it / inside) to 0.42 / 0.47 / 1.20, a 256x256 frame of a 128^3 one
//    from 58 to 31 us, a 2160p frame of a 512^3 one from 2.59 to 1.69.
//  * whether a batch lies inside the grid and the ray is asked once, of its
//    last step, as both only ever end; what is left of a ray is one batch more,
//    asked step by step.
//  * a step's masks come from one three-way minimum of the side distances' bits
//    (no NaN handling), and its voxel is kept as three counters of voxels to go,
//    each lowered by one subtract-with-borrow.
// ---------------------------------------------------------------------------
// a * b + c for a, b < 2^24, a full-rate instruction (the compiler takes a
// 64-bit multiply-add for the same expression).
__device__ __forceinline__ uint32_t mad24(uint32_t a, uint32_t b, uint32_t c) {
    uint32_t r;
    asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(b), "v"(c));
    return r;
}

// Bit of macro cell (cx, cy, cz) in a bitmask.  A bitmask holds at
// most kMaxMacroWords * 32 = 2^17 cells, so every operand and partial result
// is below 2^24 and the 24-bit multiply-add (full rate) is exact.
__device__ __forceinline__ uint32_t macro_cell(uint32_t cx, uint32_t cy, uint32_t cz, uint32_t mnx, uint32_t mny) {
    return mad24(mad24(cz, mny, cy), mnx, cx);
}

// Texel index of voxel (ux, uy, uz) in the bricked grid, 32-bit form.  Grids
// take it only when nbz * nby < 2^24 and nbx < 2^24 (else the 64-bit form;
// see fill_params), so both multiplies' operands are below 2^24.
__device__ __forceinline__ uint32_t brick_texel32(uint32_t ux, uint32_t uy, uint32_t uz, uint32_t nbx, uint32_t nby,
                                                  uint32_t in_brick) {
    return (mad24(mad24(uz >> 2, nby, uy >> 2), nbx, ux >> 2) << 6) + in_brick;
}

// One step: the axes whose side distance is the least, and that distance.
// Side distances are +0 or more (or NaN, at most one of them here), so as
// unsigned words they are ordered as the floats are, and the axes equal to the
// least are the shader's mask.
struct DdaStep {
    float t;
    bool x, y, z;
};
__device__ __forceinline__ DdaStep dda_step(f3 sd) {
    uint32_t m;
    asm("v_min3_u32 %0, %1, %2, %3" : "=v"(m) : "v"(f2u(sd.x)), "v"(f2u(sd.y)), "v"(f2u(sd.z)));
    return DdaStep{u2f(m), f2u(sd.x) == m, f2u(sd.y) == m, f2u(sd.z) == m};
}
__device__ __forceinline__ f3 dda_next(f3 sd, f3 t_delta, const DdaStep& s) {
    return mk(sd.x + (s.x ? t_delta.x : 0.0f), sd.y + (s.y ? t_delta.y : 0.0f), sd.z + (s.z ? t_delta.z : 0.0f));
}

template <bool COUNT, bool WIDE, uint32_t RUN>
__device__ __forceinline__ f3 dda_trace(const RenderParams& p, const uint32_t* __restrict__ masks, f3 ro, f3 rd,
                                        uint64_t& words) {
    f3 rrd = divv(splat(1.0f), rd);
    f3 bias = mul(rrd, ro);
    f3 box_min = neg(bias);
    f3 md = mk((float)p.view.model_dim[0], (float)p.view.model_dim[1], (float)p.view.model_dim[2]);
    f3 box_max = sub(mul(md, rrd), bias);
    float t_min = max_elem(vmin(box_min, box_max));
    float t_max = min_elem(vmax(box_min, box_max));
    if (t_min > t_max) return splat(0.0f);
    t_min = gmax(t_min, 0.0f);
    ro = add(ro, muls(rd, t_min));
    int32_t px = f2i_sat(ro.x), py = f2i_sat(ro.y), pz = f2i_sat(ro.z);
    f3 t_delta = mk(fabs_(rrd.x), fabs_(rrd.y), fabs_(rrd.z));
    f3 sgn = mk(fsign(rd.x), fsign(rd.y), fsign(rd.z));
    f3 fl = mk(__builtin_floorf(ro.x), __builtin_floorf(ro.y), __builtin_floorf(ro.z));
    f3 sd = mul(add(mul(sgn, add(sub(fl, ro), splat(0.5f))), splat(0.5f)), t_delta);
    float t = 0.0f;
    f3 total = splat(0.0f);
    const float limit = t_max - t_min;
    const uint32_t cap32 = cap32_of(p.cap);
    uint32_t it = 0;
    if (COUNT) {
        while (t < limit) {
            if (++it > cap32) break;
            bool mx = sd.x <= gmin(sd.y, sd.z);
            bool my = sd.y <= gmin(sd.z, sd.x);
            bool mz = sd.z <= gmin(sd.x, sd.y);
            t = min_elem(sd);
            ++words;
            sd = add(sd, mk(mx ? t_delta.x : 0.0f, my ? t_delta.y : 0.0f, mz ? t_delta.z : 0.0f));
        }
        return total;
    }
    const uint32_t X = p.dims[0], Y = p.dims[1], Z = p.dims[2];
    const uint32_t nbx = p.nb[0], nby = p.nb[1];
    const uint32_t ms = p.macro_shift, mnx = p.mn[0], mny = p.mn[1];
    auto texel = [&](uint32_t ux, uint32_t uy, uint32_t uz) -> uint32_t {
        const uint32_t in_brick = (ux & 3u) + ((uy & 3u) << 2) + ((uz & 3u) << 4);
        if (WIDE) return p.bricks[(((uint64_t)(uz >> 2) * nby + (uy >> 2)) * nbx + (ux >> 2)) * 64u + in_brick];
        return p.bricks[brick_texel32(ux, uy, uz, nbx, nby, in_brick)];
    };
    // a camera with two NaN coordinates: no axis ever steps, so the first
    // texel's term is the whole sum
    if (((sd.x != sd.x) + (sd.y != sd.y) + (sd.z != sd.z)) >= 2) {
        if (t < limit && (uint32_t)px < X && (uint32_t)py < Y && (uint32_t)pz < Z) {
            const uint32_t v = texel((uint32_t)px, (uint32_t)py, (uint32_t)pz);
            if (v & 0xFFFFFFu) total = add(total, muls(unorm_rgb(v), min_elem(sd)));
        }
        return total;
    }
    const bool fx = sgn.x > 0.0f, fy = sgn.y > 0.0f, fz = sgn.z > 0.0f;
    // to the first voxel inside the grid
    while (t < limit && !((uint32_t)px < X && (uint32_t)py < Y && (uint32_t)pz < Z)) {
        if (++it > cap32) return total;
        const DdaStep s = dda_step(sd);
        t = s.t;
        sd = dda_next(sd, t_delta, s);
        px += s.x ? (fx ? 1 : -1) : 0;
        py += s.y ? (fy ? 1 : -1) : 0;
        pz += s.z ? (fz ? 1 : -1) : 0;
    }
    // voxels left before the ray leaves the grid, along each axis: a counter
    // that a step lowers by its mask (one subtract-with-borrow), inside the
    // grid as long as it is above 0; the voxel is (n ^ flip) + base
    const uint32_t ux = (uint32_t)px, uy = (uint32_t)py, uz = (uint32_t)pz;
    int32_t nx = (int32_t)(fx ? X - ux : ux + 1u), ny = (int32_t)(fy ? Y - uy : uy + 1u),
            nz = (int32_t)(fz ? Z - uz : uz + 1u);
    const uint32_t flx = fx ? ~0u : 0u, fly = fy ? ~0u : 0u, flz = fz ? ~0u : 0u;
    const uint32_t bsx = fx ? X + 1u : ~0u, bsy = fy ? Y + 1u : ~0u, bsz = fz ? Z + 1u : ~0u;
    auto in_reach = [&]() {  // the macro mask at the current voxel
        const uint32_t cx = (((uint32_t)nx ^ flx) + bsx) >> ms, cy = (((uint32_t)ny ^ fly) + bsy) >> ms,
                       cz = (((uint32_t)nz ^ flz) + bsz) >> ms;
        const uint32_t bit = macro_cell(cx, cy, cz, mnx, mny);
        return ((masks[bit >> 5] >> (bit & 31u)) & 1u) != 0;
    };
    // batches of RUN steps that all lie inside the grid and the ray
    uint32_t vx[RUN], vy[RUN], vz[RUN], tex[RUN];
    float dts[RUN];
    auto take = [&](uint32_t j) {  // step j of a batch: its voxel and its length
        vx[j] = ((uint32_t)nx ^ flx) + bsx;
        vy[j] = ((uint32_t)ny ^ fly) + bsy;
        vz[j] = ((uint32_t)nz ^ flz) + bsz;
        const DdaStep s = dda_step(sd);
        dts[j] = s.t - t;
        t = s.t;
        sd = dda_next(sd, t_delta, s);
        nx -= s.x ? 1 : 0;
        ny -= s.y ? 1 : 0;
        nz -= s.z ? 1 : 0;
    };
    const uint32_t whole_cap = cap32 - RUN;
    while (it <= whole_cap) {
        const f3 sd0 = sd;
        const float t_start = t;
        const int32_t nx0 = nx, ny0 = ny, nz0 = nz;
        bool whole = false;
#pragma unroll
        for (uint32_t j = 0; j < RUN; ++j) {
            if (j == RUN - 1) whole = t < limit && min(min(nx, ny), nz) > 0;
            take(j);
        }
        const int32_t nx1 = nx, ny1 = ny, nz1 = nz;
        nx = nx0;
        ny = ny0;
        nz = nz0;
        if (!whole) {
            sd = sd0;
            t = t_start;
            break;
        }
        it += RUN;
        if (in_reach()) {
#pragma unroll
            for (uint32_t j = 0; j < RUN; ++j) tex[j] = texel(vx[j], vy[j], vz[j]);
#pragma unroll
            for (uint32_t j = 0; j < RUN; ++j)
                if (tex[j] & 0xFFFFFFu) total = add(total, muls(unorm_rgb(tex[j]), dts[j]));
        }
        nx = nx1;
        ny = ny1;
        nz = nz1;
    }
    // the rest of the ray, at most RUN steps
    if (t < limit && min(min(nx, ny), nz) > 0 && in_reach()) {
        bool valid[RUN];
#pragma unroll
        for (uint32_t j = 0; j < RUN; ++j) {
            valid[j] = t < limit && min(min(nx, ny), nz) > 0 && it + j < cap32;
            take(j);
        }
#pragma unroll
        for (uint32_t j = 0; j < RUN; ++j) tex[j] = valid[j] ? texel(vx[j], vy[j], vz[j]) : 0u;
#pragma unroll
        for (uint32_t j = 0; j < RUN; ++j)
            if (tex[j] & 0xFFFFFFu) total = add(total, muls(unorm_rgb(tex[j]), dts[j]));
    }
    return total;
}

// ---------------------------------------------------------------------------
// Octree kernels (main() of svo_naive/svo_df/esvo/svo_rope.comp)
//   TAGGED && !COUNT  fast traversals on the tagged layout (xd_svo_fast.hpp)
//   otherwise         reference-structured traversals (xd_svo_ref.hpp)
// ---------------------------------------------------------------------------
// LDS_TOP: the kernel may stage top-level child words in LDS (plain
// launches; only svo-rope's views do).  Where no view can, the traversal is
// built with no top levels at all, which drops the LDS-or-device-memory
// choice from every child-word read.
template <int TRAV, bool COUNT, bool TAGGED, bool LDS_TOP = true>
__device__ __forceinline__ f3 svo_pixel(const RenderParams& p, f3 rd, uint32_t* lds, const uint32_t* lds_top,
                                        uint64_t& words) {
    // this wavefront's stack region: two arrays of lds_slots x 64 lane-strided
    // words.  The stride is the launch's (all views of a batch share it), not
    // this tree's, so regions of different waves never overlap.
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
    uint32_t* stk_a = lds + wave * 2u * p.lds_slots * kWaveLanes + lane;
    uint32_t* stk_b = stk_a + p.lds_slots * kWaveLanes;
    const uint32_t n_top = LDS_TOP && TRAV == 4 ? p.top_nodes : 0u;  // svo-rope
    const FastSvo fs = make_fast_svo(p.cw, p.meta, p.root_tag, lds_top, n_top, p.node_count, p.depth_exact, p.table, p.table_shift, p.rope_depth,
                      p.index_mask, p.empty_tag, p.empty_start, p.leaf_base);
    if (TRAV == 2) {  // esvo
        f3 ro = add(p.cam.translation, splat(1.0f));
        float t0, t1;
        aabb_intersect(splat(1.0f), splat(2.0f), ro, rd, t0, t1);
        ro = add(ro, smul(gmax(t0, 0.0f), rd));
        if (TAGGED && !COUNT && p.stack_slots - 2u < kEsvoCellLevels) {  // 1 to kEsvoCellLevels levels
            const EsvoRay r = esvo_setup(ro, rd);
            if (esvo_cell_ray(ro, rd, r)) return fast_esvo_cells(fs, p.rec, p.stack_slots - 1u, p.cap, rd, r);
        }
        float* stk_tmax = reinterpret_cast<float*>(stk_b);
        for (uint32_t s = 0; s < p.stack_slots; ++s) {
            stk_a[s * kWaveLanes] = 0u;
            stk_tmax[s * kWaveLanes] = 0.0f;
        }
        if (TAGGED && !COUNT) return fast_esvo(fs, p.cap, p.stack_slots, ro, rd, stk_a,
                                                stk_tmax);
        if (TAGGED) return ref_esvo<COUNT>(TaggedNodes{p.cw, p.meta, p.node_count, p.index_mask, p.leaf_base}, p.cap, p.stack_slots, ro, rd, stk_a, stk_tmax,
                                           words);
        return ref_esvo<COUNT>(RawNodes{p.nodes, p.node_count}, p.cap, p.stack_slots, ro, rd, stk_a, stk_tmax, words);
    }
    const f3 ro = p.cam.translation;
    if (TRAV == 3) {  // svo-df
        if (TAGGED && !COUNT && p.rec) {
            const f3 rrd = divv(splat(1.0f), rd), bias = mul(rrd, ro);
            if (df_ray(rrd, bias)) return fast_df_rec(p.rec, p.leaf_base, p.cap, rrd, bias, stk_a, stk_b);
        }
        if (TAGGED && !COUNT)  // depth-field handling fixed per tree (a uniform choice)
            return p.depth_exact ? fast_df<true>(fs, p.cap, p.stack_slots, ro, rd, stk_a, stk_b)
                                 : fast_df<false>(fs, p.cap, p.stack_slots, ro, rd, stk_a, stk_b);
        if (TAGGED) return ref_df<COUNT>(TaggedNodes{p.cw, p.meta, p.node_count, p.index_mask, p.leaf_base}, p.cap, p.stack_slots, ro, rd, stk_a, stk_b, words);
        return ref_df<COUNT>(RawNodes{p.nodes, p.node_count}, p.cap, p.stack_slots, ro, rd, stk_a, stk_b, words);
    }
    if (TRAV == 1) {  // svo-naive
        if (TAGGED && !COUNT) return fast_naive(fs, p.rec, p.cap, ro, rd);
        if (TAGGED) return ref_naive<COUNT>(TaggedNodes{p.cw, p.meta, p.node_count, p.index_mask, p.leaf_base}, p.cap, ro, rd, words);
        return ref_naive<COUNT>(RawNodes{p.nodes, p.node_count}, p.cap, ro, rd, words);
    }
    // svo-rope
    if (TAGGED && !COUNT && p.rope_cells && rope_cell_ray(ro, rd))
        return fast_rope_cells(fs, p.rec, p.cap, ro, rd);
    if (TAGGED && !COUNT) return fast_rope(fs, p.cap, ro, rd);
    if (TAGGED) return ref_rope<COUNT>(TaggedNodes{p.cw, p.meta, p.node_count, p.index_mask, p.leaf_base}, p.cap, ro, rd, words);
    return ref_rope<COUNT>(RawNodes{p.nodes, p.node_count}, p.cap, ro, rd, words);
}

}  // namespace xd
