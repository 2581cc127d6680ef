// fg_contact.hpp -- penalty contact of one sphere against the spheres of a
// bucket grid (GPU_Kernels/K_DeviceFunctions.cu:32-159), written with the
// reference's arithmetic and contraction off.
#pragma once
#include "fg_internal.hpp"

namespace fg {
#pragma clang fp contract(off)

// One sphere of ProcessCellForcesD (K_DeviceFunctions.cu:32-106): sphere i
// at pos; for a sphere within mind = r_i + r_j + eps, F += (ks*l - kd*dot(n,
// v_j - v_i)) * n with n = (x_j - x_i)/l, l = |x_j - x_i| (the spring term
// uses the distance).  Velocities: per body (indexed by w) when w_index,
// else per sphere; none when vel is null.  A sphere's velocity enters only
// a contact term, so it is read only for spheres in contact.
//
// cut2 = mind^2 (1 + 2^-20), rounded, exceeds mind^2 (1 + 2^-21): a sphere
// with |x_j - x_i|^2 > cut2 has a distance above mind by more than two
// units in the last place of mind, so its rounded square root is not below
// mind and the exact test would reject it too.  Most spheres of a walked
// bucket are rejected by that comparison of the squared distance, without
// the square root.
__device__ __forceinline__ F3 contact_term(F3 F, const float4& pos, uint32_t i, const float4& sp, const float4& sv,
                                           float mind, float cut2, const float4* __restrict__ cvel, float ks,
                                           float kd, bool w_index, bool group, int w_group, uint32_t vlimit) {
    if (group && f2i_sat(pos.w) == w_group) return F;
    const F3 rel = sub(xyz(pos), xyz(sp));
    const float r2 = dot(rel, rel);
    if (!(r2 <= cut2)) return F;  // also NaN, which the exact test rejects as well
    const float lg = rn_sqrt(r2);  // len(rel)
    if (lg < mind) {
        float4 vel = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (cvel) {
            const uint32_t vi = w_index ? (uint32_t)f2i_sat(pos.w) : i;
            if (vi < vlimit) vel = cvel[vi];
        }
        const F3 n = divs(rel, lg);
        const F3 rv = sub(xyz(vel), xyz(sv));
        F = add(F, mul(ks * lg - kd * dot(n, rv), n));
    }
    return F;
}

// ProcessCellForcesD over the sorted range [s0, e_raw) of one bucket
// (spheres in order; two positions are loaded at a time).
__device__ __forceinline__ F3 contact_range(const float4& sp, const float4& sv, float sr, float cr,
                                            const float4* __restrict__ cpos, const float4* __restrict__ cvel,
                                            uint32_t s0, uint32_t e_raw, float ks, float kd, bool w_index,
                                            bool group, int w_group, float eps, uint32_t limit, uint32_t vlimit) {
    F3 F = f3(0.0f, 0.0f, 0.0f);
    const float mind = sr + cr + eps;
    const float cut2 = rn_mul(rn_mul(mind, mind), 0x1.00001p+0f);
    if (s0 != kEmpty) {
        const uint32_t e = min(e_raw, limit);
        uint32_t i = s0;
        for (; i + 1 < e; i += 2) {
            const float4 p0 = cpos[i], p1 = cpos[i + 1];
            F = contact_term(F, p0, i, sp, sv, mind, cut2, cvel, ks, kd, w_index, group, w_group, vlimit);
            F = contact_term(F, p1, i + 1, sp, sv, mind, cut2, cvel, ks, kd, w_index, group, w_group, vlimit);
        }
        if (i < e)
            F = contact_term(F, cpos[i], i, sp, sv, mind, cut2, cvel, ks, kd, w_index, group, w_group, vlimit);
    }
    return F;
}

// Bucket of stencil offset (x,y,z) around sp, or kEmpty for a LINEAR cell
// outside the grid.
__device__ __forceinline__ uint32_t contact_key(const float4& sp, const CellXYZ& c, int x, int y, int z,
                                                const GridDesc& g) {
    if (g.mode == FG_KEY_REF_XOR) {
        const float ox = g.cs.x * (float)x, oy = g.cs.y * (float)y, oz = g.cs.z * (float)z;
        return g.key_base + hash_ref_xor(sp.x + ox, sp.y + oy, sp.z + oz, g.cs.x, g.cs.y, g.cs.z, g.nb);
    }
    const int a = c.x + x, b = c.y + y, d = c.z + z;
    if (a < 0 || b < 0 || d < 0 || a >= g.dims.x || b >= g.dims.y || d >= g.dims.z) return kEmpty;
    return g.key_base + grid_linear_key(a, b, d, g);
}

// The reference hash is an XOR of per-axis products, and each axis term
// depends only on that coordinate and its stencil offset.  For the stencil
// (1,1,1) the three terms per axis are computed once (9 IEEE divisions
// instead of 81) and combined per cell; every key is the one hash_ref_xor
// gives for that cell.
struct XorAxisTerms {
    uint32_t x[3], y[3], z[3];
};
__device__ __forceinline__ uint32_t xor_axis_term(float p, float cs, float off, uint32_t prime) {
    return (uint32_t)f2i_sat(rn_div(rn_add(p + cs * off, 5000.0f), cs)) * prime;
}
__device__ __forceinline__ XorAxisTerms xor_axis_terms(const float4& sp, const GridDesc& g) {
    XorAxisTerms t;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const float o = (float)(k - 1);
        t.x[k] = xor_axis_term(sp.x, g.cs.x, o, 73856093u);
        t.y[k] = xor_axis_term(sp.y, g.cs.y, o, 19349663u);
        t.z[k] = xor_axis_term(sp.z, g.cs.z, o, 83492791u);
    }
    return t;
}
__device__ __forceinline__ uint32_t sel3(const uint32_t (&v)[3], int k) {
    return k < 0 ? v[0] : (k > 0 ? v[2] : v[1]);
}
// The bucket of hash h (a mask instead of the division where the table has a
// power of two of buckets).
__device__ __forceinline__ uint32_t xor_bucket(uint32_t h, const GridDesc& g) {
    return g.key_base + ((g.nb & (g.nb - 1u)) == 0u ? h & (g.nb - 1u) : h % g.nb);
}
__device__ __forceinline__ uint32_t xor_key(const XorAxisTerms& t, int x, int y, int z, const GridDesc& g) {
    return xor_bucket(sel3(t.x, x) ^ sel3(t.y, y) ^ sel3(t.z, z), g);
}

// ProcessCollisionForcesD, K_DeviceFunctions.cu:113-159: the (2r+1)^3
// stencil in z, y, x order around one lane's sphere, on a grid keyed with the
// reference hash, which rehashes x + k*cs.
__device__ __forceinline__ F3 contact_stencil(const float4& sp, const float4& sv, float sr,
                                              const float4* __restrict__ cpos, const float4* __restrict__ cvel,
                                              float cr, float ks, float kd, int3 rel,
                                              const uint32_t* __restrict__ start, const uint32_t* __restrict__ end,
                                              const GridDesc& g, bool w_index, float eps, uint32_t limit,
                                              uint32_t vlimit) {
    F3 F = f3(0.0f, 0.0f, 0.0f);
    GridDesc gg = g;
    gg.mode = FG_KEY_REF_XOR;
    const bool unit = rel.x == 1 && rel.y == 1 && rel.z == 1;
    XorAxisTerms t{};
    if (unit) t = xor_axis_terms(sp, gg);
    for (int z = -rel.z; z <= rel.z; z++)
        for (int y = -rel.y; y <= rel.y; y++)
            for (int x = -rel.x; x <= rel.x; x++) {
                const uint32_t key = unit ? xor_key(t, x, y, z, gg) : contact_key(sp, CellXYZ{0, 0, 0}, x, y, z, gg);
                const uint32_t s0 = start[key];
                F = add(F, contact_range(sp, sv, sr, cr, cpos, cvel, s0, s0 != kEmpty ? end[key] : 0u, ks, kd, w_index,
                                         false, 0, eps, limit, vlimit));
            }
    return F;
}

// Force on a fluid particle from one body grid (K_FluidSim.cu:372-386);
// zero outside the expanded sphere bounds, where no contact is possible.
__device__ __forceinline__ F3 fluid_body_contact(const float4& pos, const float4& vel, const BodyContact& bc) {
    if (bc.aabb) {
        const float4 lo = bc.aabb[0], hi = bc.aabb[1];
        if (pos.x < lo.x || pos.y < lo.y || pos.z < lo.z || pos.x > hi.x || pos.y > hi.y || pos.z > hi.z)
            return f3(0.0f, 0.0f, 0.0f);
    }
    // body grids are keyed with the reference hash (body_grid in fg_rigid.hip)
    return contact_stencil(pos, vel, bc.fluid_radius, bc.pos, bc.vel, bc.body_radius, bc.ks, bc.kd, bc.relation,
                           bc.start, bc.end, bc.grid, bc.vel != nullptr, bc.eps, bc.count, bc.nvel);
}

// Memory that one wavefront's groups of kContactLanes lanes share in
// contact_stencil_lanes, per group: the non-empty cells of a batch (first
// sphere and count), the spheres within reach (index and cell), one
// round's terms by component with their cells, and the axis terms of the
// hash.  The odd row lengths keep the
// groups' rows in different banks.
constexpr uint32_t kContactLanes = 8;
struct ContactWave {
    static constexpr uint32_t kCells = 32, kHits = 32;
    uint2 cell[64 / kContactLanes][kCells + 1];
    uint2 hit[64 / kContactLanes][kHits + 1];
    float4 term[64 / kContactLanes][3][2];
    uint4 cell_of[64 / kContactLanes][2];
    uint32_t axis[64 / kContactLanes][kContactLanes + 1];
};

// Orders a wavefront's LDS stores before its other lanes' loads (and loads
// before the next stores): the lanes of one wavefront need no workgroup
// barrier.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// contact_stencil (on a LINEAR grid too: its cells outside the grid are
// skipped, K_DeviceFunctions.cu:113-159) by a group of
// kContactLanes = 8 consecutive lanes of a wavefront (sub: the lane's index
// in its group; every lane of the group active and holding the same sphere).
//
// The walk is bound by chains of dependent loads (cell start, spheres,
// velocity) and by work done for few lanes, so it is cut into passes that
// keep the group's lanes together:
//   1. every lane finds four cells, their starts and ends in flight together,
//      and the non-empty cells are listed in stencil order;
//   2. cell after cell, eight spheres at a time, are tested by squared
//      distance (the next eight already loading), and those within reach are
//      listed in order;
//   3. the listed spheres' terms are computed eight at a time, and one lane
//      per component adds them in order: each cell into a sum of its own from
//      zero, each cell's sum to the total.
// A full list is worked off and the walk goes on, so any cell length is
// served, and stencils of more than 32 cells take their cells by 32.  The
// additions are contact_stencil's, in its order, without those of zeros: a
// running sum that starts at +0 is never -0 under round-to-nearest, so the
// skipped ones change no bit.
//
// 1,048,576 particles, 112k of them inside the bounds of a torus or a post
// (33 spheres to test and 4 in contact each on average), finish pass:
// 104 us with two lanes a particle that walked their cells one after another,
// 58 us so; body forces of 19,936 spheres (108 to test, 9 in contact): 29 us
// and 24 us.  What bounds it now: the instructions of the walk, about 60 for
// each pass of eight spheres.
__device__ __forceinline__ F3 contact_stencil_lanes(const float4& sp, const float4& sv, float sr,
                                                    const float4* __restrict__ cpos, const float4* __restrict__ cvel,
                                                    float cr, float ks, float kd, int3 rel,
                                                    const uint32_t* __restrict__ start,
                                                    const uint32_t* __restrict__ end, const GridDesc& g,
                                                    bool w_index, bool group, int w_group, float eps, uint32_t limit,
                                                    uint32_t vlimit, uint32_t sub, ContactWave& W) {
    constexpr uint32_t LP = kContactLanes, kPer = ContactWave::kCells / LP;
    const uint32_t lane = __lane_id(), first = lane & ~(LP - 1u), gr = lane / LP, below = (1u << sub) - 1u;
    auto group_bits = [first](bool b) { return (uint32_t)(__ballot(b) >> first) & ((1u << LP) - 1u); };
    const float mind = sr + cr + eps;
    const float cut2 = rn_mul(rn_mul(mind, mind), 0x1.00001p+0f);
    const CellXYZ c = g.mode == FG_KEY_LINEAR ? grid_cell(sp.x, sp.y, sp.z, g) : CellXYZ{0, 0, 0};
    // (an axis of negative width leaves no cell)
    const int nx = 2 * rel.x + 1, ny = 2 * rel.y + 1, cells = (rel.x | rel.y | rel.z) < 0 ? 0 : nx * ny * (2 * rel.z + 1);
    const bool unit = rel.x == 1 && rel.y == 1 && rel.z == 1;
    const bool xor_unit = unit && g.mode == FG_KEY_REF_XOR;
    const float csx = g.cs.x, csy = g.cs.y, csz = g.cs.z;
    if (xor_unit) {  // the nine axis terms of the hash: one a lane, the last on every lane
        wave_lds_sync();
        W.axis[gr][sub] = xor_axis_term(sub < 3u ? sp.x : (sub < 6u ? sp.y : sp.z), sub < 3u ? csx : (sub < 6u ? csy : csz),
                                        (float)((int)(sub % 3u) - 1),
                                        sub < 3u ? 73856093u : (sub < 6u ? 19349663u : 83492791u));
        if (sub == 0u) W.axis[gr][LP] = xor_axis_term(sp.z, csz, 1.0f, 83492791u);
        wave_lds_sync();
    }

    float total = 0.0f, part = 0.0f;  // of component sub, on lanes 0..2
    uint32_t cell = 0, hits = 0;      // part's cell; spheres listed (the same on a group's lanes)
    auto add_listed = [&]() {
        wave_lds_sync();
        for (uint32_t t0 = 0; __any(t0 < hits); t0 += LP) {
            F3 f = f3(0.0f, 0.0f, 0.0f);
            uint2 q = make_uint2(0u, 0u);
            if (t0 < hits) {
                q = W.hit[gr][min(t0 + sub, hits - 1u)];  // lanes past the end: the last one's cell and +0
                if (t0 + sub < hits)
                    f = contact_term(f, cpos[q.x], q.x, sp, sv, mind, cut2, cvel, ks, kd, w_index, group, w_group,
                                     vlimit);
            }
            float* const term = reinterpret_cast<float*>(W.term[gr]);
            term[sub] = f.x;
            term[LP + sub] = f.y;
            term[2 * LP + sub] = f.z;
            reinterpret_cast<uint32_t*>(W.cell_of[gr])[sub] = q.y;
            wave_lds_sync();
            if (t0 < hits && sub < 3u) {
                const float4 a = W.term[gr][sub][0], b = W.term[gr][sub][1];
                const uint4 ca = W.cell_of[gr][0], cb = W.cell_of[gr][1];
                const float v[LP] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
                const uint32_t k[LP] = {ca.x, ca.y, ca.z, ca.w, cb.x, cb.y, cb.z, cb.w};
#pragma unroll
                for (uint32_t u = 0; u < LP; u++) {
                    if (k[u] != cell) {
                        total = rn_add(total, part);
                        part = 0.0f;
                        cell = k[u];
                    }
                    part = rn_add(part, v[u]);
                }
            }
            wave_lds_sync();  // the reads before the next round's terms
        }
        hits = 0;
    };

    for (int b = 0; b < cells; b += (int)ContactWave::kCells) {
        uint32_t s[kPer], m[kPer];
#pragma unroll
        for (uint32_t r = 0; r < kPer; r++) {
            const int k = b + (int)(sub * kPer + r);
            s[r] = kEmpty;
            m[r] = 0;
            if (k >= cells) continue;
            uint32_t key;
            if (xor_unit)
                key = xor_bucket(W.axis[gr][k % 3] ^ W.axis[gr][3 + (k / 3) % 3] ^ W.axis[gr][6 + k / 9], g);
            else if (unit)
                key = contact_key(sp, c, k % 3 - 1, (k / 3) % 3 - 1, k / 9 - 1, g);
            else
                key = contact_key(sp, c, k % nx - rel.x, (k / nx) % ny - rel.y, k / (nx * ny) - rel.z, g);
            if (key != kEmpty) {  // a LINEAR cell outside the grid adds nothing
                s[r] = start[key];
                m[r] = end[key];
            }
        }
        uint32_t at = 0, count = 0;
#pragma unroll
        for (uint32_t r = 0; r < kPer; r++) {
            const uint32_t e = min(m[r], limit);
            m[r] = s[r] != kEmpty && s[r] < e ? e - s[r] : 0u;
            const uint32_t bits = group_bits(m[r] != 0u);
            at += __popc(bits & below);
            count += __popc(bits);
        }
        wave_lds_sync();  // the last batch's cells have been read
#pragma unroll
        for (uint32_t r = 0; r < kPer; r++)
            if (m[r] != 0u) W.cell[gr][at++] = make_uint2(s[r], m[r]);
        wave_lds_sync();

        // spheres [off, off + 8) of cell j; the next eight are loaded before these are tested
        uint32_t j = 0, off = 0;
        uint2 cur = count ? W.cell[gr][0] : make_uint2(0u, 0u);
        float4 p = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (sub < cur.y) p = cpos[cur.x + sub];
        for (;;) {
            const bool more = __any(j < count);
            if (__any(hits > (more || b + (int)ContactWave::kCells < cells ? ContactWave::kHits - LP : 0u))) add_listed();
            if (!more) break;
            uint32_t nj = j, noff = off + LP;
            uint2 nxt = cur;
            if (noff >= cur.y) {
                nj = j + 1u;
                noff = 0;
                nxt = nj < count ? W.cell[gr][nj] : make_uint2(0u, 0u);
            }
            float4 np = p;
            if (noff + sub < nxt.y) np = cpos[nxt.x + noff + sub];
            bool hit = off + sub < cur.y;
            if (hit) {
                const F3 d = f3(p.x - sp.x, p.y - sp.y, p.z - sp.z);
                hit = dot(d, d) <= cut2 && !(group && f2i_sat(p.w) == w_group);
            }
            if (__any(hit)) {
                const uint32_t bits = group_bits(hit);
                if (hit)
                    W.hit[gr][hits + __popc(bits & below)] =
                        make_uint2(cur.x + off + sub, (uint32_t)b + j);
                hits += __popc(bits);
            }
            j = nj;
            off = noff;
            cur = nxt;
            p = np;
        }
    }
    total = rn_add(total, part);
    return f3(__shfl(total, (int)first), __shfl(total, (int)first + 1), __shfl(total, (int)first + 2));
}

// contact_stencil_lanes with a cell a lane: lane sub walks cells sub, sub + 8,
// ... of the z, y, x stencil order by itself, each into a sum of its own from
// zero, and after each round of eight the group adds the round's sums in cell
// order, without those of zeros.  The same bits.  For a wide stencil, most of
// whose cells are out of reach: a cell of eight spheres costs a lane of its own
// less than a pass of the whole group.
__device__ __forceinline__ F3 contact_stencil_apart(const float4& sp, const float4& sv, float sr,
                                                    const float4* __restrict__ cpos, const float4* __restrict__ cvel,
                                                    float cr, float ks, float kd, int3 rel,
                                                    const uint32_t* __restrict__ start,
                                                    const uint32_t* __restrict__ end, const GridDesc& g, float eps,
                                                    uint32_t limit, uint32_t vlimit, uint32_t sub) {
    F3 F = f3(0.0f, 0.0f, 0.0f);
    const CellXYZ c = g.mode == FG_KEY_LINEAR ? grid_cell(sp.x, sp.y, sp.z, g) : CellXYZ{0, 0, 0};
    const int nx = 2 * rel.x + 1, ny = 2 * rel.y + 1, cells = (rel.x | rel.y | rel.z) < 0 ? 0 : nx * ny * (2 * rel.z + 1);
    const uint32_t first = __lane_id() & ~(kContactLanes - 1u);
    for (int r0 = 0; r0 < cells; r0 += (int)kContactLanes) {
        const int k = r0 + (int)sub;
        F3 part = f3(0.0f, 0.0f, 0.0f);
        if (k < cells) {
            const uint32_t key = contact_key(sp, c, k % nx - rel.x, (k / nx) % ny - rel.y, k / (nx * ny) - rel.z, g);
            if (key != kEmpty) {
                const uint32_t s0 = start[key], e = end[key];
                part = contact_range(sp, sv, sr, cr, cpos, cvel, s0, s0 != kEmpty ? e : 0u, ks, kd, false, false, 0, eps,
                                     limit, vlimit);
            }
        }
        const uint64_t nonzero = __ballot(part.x != 0.0f || part.y != 0.0f || part.z != 0.0f);
        uint32_t m = (uint32_t)(nonzero >> first) & ((1u << kContactLanes) - 1u);
        while (m) {
            const int src = (int)first + __ffs((int)m) - 1;
            m &= m - 1u;
            F = add(F, f3(__shfl(part.x, src), __shfl(part.y, src), __shfl(part.z, src)));
        }
    }
    return F;
}

// fluid_body_contact by a group of lanes (contact_stencil_lanes).
__device__ __forceinline__ F3 contact_cells(const float4& pos, const float4& vel, const BodyContact& bc, uint32_t sub,
                                            ContactWave& W) {
    if (bc.aabb) {
        const float4 lo = bc.aabb[0], hi = bc.aabb[1];
        if (pos.x < lo.x || pos.y < lo.y || pos.z < lo.z || pos.x > hi.x || pos.y > hi.y || pos.z > hi.z)
            return f3(0.0f, 0.0f, 0.0f);
    }
    GridDesc g = bc.grid;
    g.mode = FG_KEY_REF_XOR;  // body grids are keyed with the reference hash (body_grid in fg_rigid.hip)
    return contact_stencil_lanes(pos, vel, bc.fluid_radius, bc.pos, bc.vel, bc.body_radius, bc.ks, bc.kd, bc.relation,
                                 bc.start, bc.end, g, bc.vel != nullptr, false, 0, bc.eps, bc.count, bc.nvel, sub, W);
}

// External force of K_FluidSim.cu:369-386: static grid first, then the
// dynamic grid, summed from zero.
__device__ __forceinline__ F3 fluid_external(const float4& pos, const float4& vel, const Contacts& c) {
    F3 e = f3(0.0f, 0.0f, 0.0f);
    if (c.st.enabled) e = add(e, fluid_body_contact(pos, vel, c.st));
    if (c.dyn.enabled) e = add(e, fluid_body_contact(pos, vel, c.dyn));
    return e;
}

#pragma clang fp contract(fast)
}  // namespace fg
