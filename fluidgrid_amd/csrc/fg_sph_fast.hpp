// fg_sph_fast.hpp -- per-particle SPH work shared by the single-fluid
// kernels (fg_sph.hip) and the batched-scene kernels (fg_batch.hip):
//  * acceleration after gravity, walls, body contact and clamp, and the
//    velocity/position write-back (reference arithmetic, contraction off);
//  * the fast LINEAR density and force passes over the 9 stencil rows.
#pragma once
#include <cstddef>

#include "fg_contact.hpp"
#include "fg_internal.hpp"
#include "fg_walls.hpp"

namespace fg {

#pragma clang fp contract(off)

// Walls and clamp of K_FluidSim.cu:293-303 applied to the acceleration
// `total` (pair sum times mass, gravity and any body contact).
__device__ __forceinline__ F3 walls_and_clamp(F3 total, const float4& pos, const float4& vel,
                                              const fg_common_fluid_params& cp) {
    F3 wall = walls_no_penetration(xyz(pos), xyz(vel), cp);
    wall = add(wall, walls_no_slip(xyz(pos), xyz(vel), cp));
    total = add(total, wall);
    const float speed = len(total);
    if (speed > cp.velocity_limit) {
        const float t = cp.velocity_limit / speed;
        total = mul(total, t);
    }
    return total;
}

// Acceleration after gravity, walls and clamp (K_FluidSim.cu:287-303), from
// the pair sum `internal`.  NO_CONTACT: the caller knows the particle lies
// outside every body grid's bounds, where fluid_external is exactly +0.
template <bool COUPLED, bool NO_CONTACT = false>
__device__ __forceinline__ F3 finish_accel(F3 internal, float m, const float4& pos, const float4& vel,
                                           const fg_common_fluid_params& cp, const Contacts& bc) {
    const F3 g = f3(cp.global_external_force.x, cp.global_external_force.y, cp.global_external_force.z);
    F3 total = add(mul(internal, m), g);
    // K_FluidSim.cu:389-390: body contact forces are added after the mass
    // factor (the uncoupled kernel adds nothing here).
    if (COUPLED && bc.coupled) total = add(total, NO_CONTACT ? f3(0.0f, 0.0f, 0.0f) : fluid_external(pos, vel, bc));
    return walls_and_clamp(total, pos, vel, cp);
}

// The same with the contact term `ext` computed by the caller (added when
// `coupled`, as fluid_external is above).
__device__ __forceinline__ F3 finish_accel_ext(F3 internal, float m, const float4& pos, const float4& vel,
                                               const fg_common_fluid_params& cp, bool coupled, F3 ext) {
    const F3 g = f3(cp.global_external_force.x, cp.global_external_force.y, cp.global_external_force.z);
    F3 total = add(mul(internal, m), g);
    if (coupled) total = add(total, ext);
    return walls_and_clamp(total, pos, vel, cp);
}

// Whether body contact can act on a particle at pos: it lies inside the
// expanded bounds of an enabled body grid (or the grid has none), the test
// with which fluid_body_contact skips its walk.
__device__ __forceinline__ bool contact_possible(const float4& pos, const Contacts& c) {
    auto inside = [&](const BodyContact& b) -> bool {
        if (!b.enabled) return false;
        if (!b.aabb) return true;
        const float4 lo = b.aabb[0], hi = b.aabb[1];
        return !(pos.x < lo.x || pos.y < lo.y || pos.z < lo.z || pos.x > hi.x || pos.y > hi.y || pos.z > hi.z);
    };
    return inside(c.st) || inside(c.dyn);
}

__device__ __forceinline__ void defer_particle(const DeferredContact& d, uint32_t i, F3 internal) {
    d.acc[i] = make_float4(internal.x, internal.y, internal.z, 0.0f);
    // one atomic per wavefront: the deferring lanes take consecutive slots
    const uint64_t lanes = __ballot(1);
    const uint32_t leader = (uint32_t)__ffsll((long long)lanes) - 1u;
    uint32_t base = 0;
    if (__lane_id() == leader) base = atomicAdd(d.count, (uint32_t)__popcll(lanes));
    base = (uint32_t)__shfl((int)base, (int)leader);
    const uint32_t lane = __lane_id();
    const uint64_t below = lane == 0 ? 0ull : (lanes & ((~0ull) >> (64 - lane)));
    d.list[base + (uint32_t)__popcll(below)] = i;
}

// vel[id] = v + a*dt, and optionally pos[id] = p + vel[id]*(dt/s) where
// p.w > 0 (K_FluidSim.cu:306-307 then :433-438).
__device__ __forceinline__ void write_back(uint32_t o, uint32_t n, const float4& pos, const float4& vel, F3 a,
                                           const fg_common_fluid_params& cp, float4* __restrict__ vout,
                                           float4* __restrict__ pout) {
    if (o >= n) return;
    const F3 dv = mul(a, cp.deltaTimeIntegration);
    const float4 nv = make_float4(vel.x + dv.x, vel.y + dv.y, vel.z + dv.z, vel.w + 0.0f);
    vout[o] = nv;
    if (pout && pos.w > 0.0f) {
        const float q = cp.deltaTimeIntegration / cp.simulation_scale;
        pout[o] = make_float4(pos.x + nv.x * q, pos.y + nv.y * q, pos.z + nv.z * q, pos.w + nv.w * q);
    }
}

#pragma clang fp contract(fast)

// ---------------------------------------------------------------------------
// Fast LINEAR kernels
// ---------------------------------------------------------------------------

// Per-particle view of the 3x3 stencil rows.  A row is the x-run of cells
// cx-1..cx+1 at (cy+dy, cz+dz); its particles are sorted[row.begin, row.end).
struct RowWalker {
    float gx_lo, gx_hi;  // squared scaled distance to the x-neighbour cells
    float gy_lo, gy_hi;  // ... to the y-neighbour slabs (0 for the own slab)
    float gz_lo, gz_hi;  // ... to the z-neighbour slabs
    int cx, cy, cz;
};

__device__ __forceinline__ float sq(float v) { return v * v; }

__device__ __forceinline__ RowWalker make_rows(const float4& p, const fg_common_fluid_params& cp) {
    RowWalker w;
    const CellXYZ c = linear_cell(p.x, p.y, p.z, cp);
    w.cx = c.x;
    w.cy = c.y;
    w.cz = c.z;
    const float s = cp.simulation_scale;
    // Lower bounds of the distance from p to the neighbouring cells along
    // each axis (zero when p lies outside its own, clamped, cell).
    const float lx = cp.volume_min.x + (float)c.x * cp.cell_size.x, hx = lx + cp.cell_size.x;
    const float ly = cp.volume_min.y + (float)c.y * cp.cell_size.y, hy = ly + cp.cell_size.y;
    const float lz = cp.volume_min.z + (float)c.z * cp.cell_size.z, hz = lz + cp.cell_size.z;
    w.gx_lo = sq(fmaxf(0.0f, p.x - lx) * s);
    w.gx_hi = sq(fmaxf(0.0f, hx - p.x) * s);
    w.gy_lo = sq(fmaxf(0.0f, p.y - ly) * s);
    w.gy_hi = sq(fmaxf(0.0f, hy - p.y) * s);
    w.gz_lo = sq(fmaxf(0.0f, p.z - lz) * s);
    w.gz_hi = sq(fmaxf(0.0f, hz - p.z) * s);
    return w;
}

// Sorted range of row (dy,dz) after culling, in two halves so that a row's
// loads can be issued a row ahead (row_fetch) and used later (row_finish).
// The grid's buckets start at key_base of the key space (0 for a single
// fluid; the scene's first bucket in a batch).  `cut` is h^2 enlarged by a
// small margin so that rounding in the cell bounds can never drop a pair
// with r < h.
struct RowFetch {
    uint32_t s0, s1, e1;  // start of the first cell, start and end of the last
    bool ok;              // the row is not culled (and s0, s1, e1 are loaded)
};

// The row's cells cx-1..cx+1 after culling by distance, as keys k0..k1;
// false for a culled row.
__device__ __forceinline__ bool row_keys(const RowWalker& w, int dy, int dz, float cut,
                                         const fg_common_fluid_params& cp, uint32_t key_base, uint32_t& k0,
                                         uint32_t& k1) {
    const int cy = w.cy + dy, cz = w.cz + dz;
    if (cy < 0 || cz < 0 || cy >= cp.bucket_size.y || cz >= cp.bucket_size.z) return false;
    // selects, not an array indexed by the row: the row loops are not always
    // unrolled, and an indexed array would live in scratch memory
    const float gy = dy < 0 ? w.gy_lo : (dy > 0 ? w.gy_hi : 0.0f);
    const float gz = dz < 0 ? w.gz_lo : (dz > 0 ? w.gz_hi : 0.0f);
    const float gyz = gy + gz;
    if (gyz >= cut) return false;
    const bool useL = w.cx > 0 && gyz + w.gx_lo < cut;                      // cell cx-1
    const bool useR = w.cx + 1 < cp.bucket_size.x && gyz + w.gx_hi < cut;  // cell cx+1
    const uint32_t kb = key_base + linear_key(0, cy, cz, cp) + (uint32_t)w.cx;
    k0 = useL ? kb - 1u : kb;
    k1 = useR ? kb + 1u : kb;
    return true;
}

// The row's particles are sorted[start[k0], end[k1]) when its end cells are
// occupied, as in the bulk of the fluid: three loads in one round trip.
__device__ __forceinline__ RowFetch row_fetch(const RowWalker& w, int dy, int dz, float cut,
                                              const fg_common_fluid_params& cp, uint32_t key_base,
                                              const uint32_t* __restrict__ start, const uint32_t* __restrict__ end) {
    RowFetch f{kEmpty, kEmpty, 0u, false};
    uint32_t k0, k1;
    if (row_keys(w, dy, dz, cut, cp, key_base, k0, k1)) {
        f.s0 = start[k0];
        f.s1 = start[k1];
        f.e1 = end[k1];
        f.ok = true;
    }
    return f;
}

// The range from the fetched loads; when an end cell is empty, the first
// occupied cell from the left and the last from the right bound it (end[]
// of an empty cell is stale and unused).  Returns false when empty.
__device__ __forceinline__ bool row_finish(const RowFetch& f, const RowWalker& w, int dy, int dz, float cut,
                                           const fg_common_fluid_params& cp, uint32_t key_base,
                                           const uint32_t* __restrict__ start, const uint32_t* __restrict__ end,
                                           uint32_t n, uint32_t& rb, uint32_t& re) {
    if (!f.ok) return false;
    if (f.s0 != kEmpty && f.s1 != kEmpty) {
        rb = f.s0;
        re = min(f.e1, n);
        return rb < re;
    }
    uint32_t k0 = 0, k1 = 0;
    row_keys(w, dy, dz, cut, cp, key_base, k0, k1);
    uint32_t b = kEmpty, e = 0;
    for (uint32_t k = k0; k <= k1; k++) {
        const uint32_t sk = start[k];
        if (sk != kEmpty) {
            if (b == kEmpty) b = sk;
            e = end[k];
        }
    }
    if (b == kEmpty) return false;
    rb = b;
    re = min(e, n);
    return rb < re;
}

__device__ __forceinline__ bool row_range(const RowWalker& w, int dy, int dz, float cut,
                                          const fg_common_fluid_params& cp, uint32_t key_base,
                                          const uint32_t* __restrict__ start, const uint32_t* __restrict__ end,
                                          uint32_t n, uint32_t& rb, uint32_t& re) {
    return row_finish(row_fetch(w, dy, dz, cut, cp, key_base, start, end), w, dy, dz, cut, cp, key_base, start,
                      end, n, rb, re);
}

// Neighbour bitmasks: for each of the 9 stencil rows of a particle, bit k of
// masks[row * n + i] is set when sorted particle rowBegin + k lies within h.
// Rows longer than 64 particles are not encoded and are re-tested.
constexpr uint32_t kRowMaskBits = 64;

// After the 9 row masks, at the next 256-byte boundary, the neighbour records
// the force pass reads for every neighbour j: two float4 per particle,
// (x_j, y_j, z_j, 1/rho_j) and (vx_j, vy_j, vz_j, p_j/rho_j), all from the
// sorted arrays.  One 32-byte record takes two 16-byte loads from one cache
// line, where position, velocity and (1/rho, p/rho) read from three arrays
// took three loads touching three lines.
__host__ __device__ __forceinline__ size_t nbr_record_offset(uint32_t n) {
    return ((size_t)9 * sizeof(unsigned long long) * n + 255) & ~(size_t)255;
}
__device__ __forceinline__ float4* nbr_records(unsigned long long* masks, uint32_t n) {
    return reinterpret_cast<float4*>(reinterpret_cast<char*>(masks) + nbr_record_offset(n));
}
__device__ __forceinline__ const float4* nbr_records(const unsigned long long* masks, uint32_t n) {
    return reinterpret_cast<const float4*>(reinterpret_cast<const char*>(masks) + nbr_record_offset(n));
}

// Then, from 256-byte boundaries, a u16 list count per particle and the lists
// of the tiled passes (kListMax u16 per particle, in 16-byte groups).
constexpr uint32_t kListMax = 64;
__host__ __device__ __forceinline__ size_t nbr_align256(size_t x) { return (x + 255) & ~(size_t)255; }
__host__ __device__ __forceinline__ size_t nbr_count_offset(uint32_t n) {
    return nbr_align256(nbr_record_offset(n) + 2 * 16 * (size_t)n);
}
__host__ __device__ __forceinline__ size_t nbr_list_offset(uint32_t n) {
    return nbr_align256(nbr_count_offset(n) + 2 * (size_t)n);
}

// The untiled passes use the list area for the deferred-contact list (its
// first 20 bytes per particle) and, after it, for the row runs that the
// density pass leaves for the force pass.  The lanes of a wavefront are 64
// consecutive sorted particles, so for each stencil row the union of their
// candidate ranges is one short run of sorted indices:
//   runs[18 w + row]     first sorted index of wavefront w's run in the row
//   runs[18 w + 9 + row] its length (kRunLength; 0 when no lane has the row),
//                        with kRunWide when a lane has more than 32
//                        candidates, kRunLong when one has more than 64,
//                        which its mask does not hold, and kRunFar, and no
//                        length, when the run is too long (kRunMax,
//                        kRunSparse): its lanes read their rows from memory
//   offs[64 (9 w + row) + lane]  the lane's first candidate, from the run's first
// A force pass that has them looks up cells for such rows only.  Both passes agree on the
// wavefronts: sorted particles 64 w .. 64 w + 63, all present (the last one
// padded by inactive lanes in a single fluid).  About 19 bytes per particle,
// which the list area holds from 64 particles on.
constexpr uint32_t kRunWords = 18;
constexpr uint32_t kRunLength = 0xFFFFu;
constexpr uint32_t kRunMax = 2047u;  // longest run
// A run above kRunSparse that is also longer than kRunSpread times what any lane
// may read of it is not staged: a wavefront of a few particles far apart, beside
// or above a pool, would stage thousands of records for a few neighbours a lane,
// and the kernel wait for it (32 splashing dam breaks, 729,000 particles:
// density 86 us, forces 85 us with every run up to kRunMax staged, 76 and 67 so).
// Where cells are full, long runs are read by most lanes and worth staging, and
// up to 640 the row costs less staged than looked up again (with 160, forces of
// 500,000 particles 50 against 47 us, a tenth of them spray).
constexpr uint32_t kRunSparse = 640u, kRunSpread = 4u;
constexpr uint32_t kRunWide = 0x10000u;
constexpr uint32_t kRunLong = 0x20000u;
constexpr uint32_t kRunFar = 0x40000u;
constexpr uint32_t kRunLookup = 0x80000u;  // (not stored) lanes look their range up: WaveCells does not hold it
constexpr uint32_t kRunMinParticles = 64;
__host__ __device__ __forceinline__ size_t nbr_runs_offset(uint32_t n) {
    return nbr_align256(nbr_list_offset(n) + 20 * (size_t)n);
}
__host__ __device__ __forceinline__ size_t nbr_offs_offset(uint32_t n) {
    return nbr_runs_offset(n) + sizeof(uint32_t) * kRunWords * (((size_t)n + 63) / 64);
}
__device__ __forceinline__ uint32_t* nbr_runs(unsigned long long* masks, uint32_t n) {
    return reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(masks) + nbr_runs_offset(n));
}
__device__ __forceinline__ const uint32_t* nbr_runs(const unsigned long long* masks, uint32_t n) {
    return reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(masks) + nbr_runs_offset(n));
}
__device__ __forceinline__ uint16_t* nbr_offs(unsigned long long* masks, uint32_t n) {
    return reinterpret_cast<uint16_t*>(reinterpret_cast<char*>(masks) + nbr_offs_offset(n));
}
__device__ __forceinline__ const uint16_t* nbr_offs(const unsigned long long* masks, uint32_t n) {
    return reinterpret_cast<const uint16_t*>(reinterpret_cast<const char*>(masks) + nbr_offs_offset(n));
}

// The host's note of what a neighbour buffer holds (fg_sph.hip).
void note_nbr_format(const void* masks, uint32_t n, bool tiled);
bool nbr_has_runs(const void* masks, uint32_t n);

// xyz of a float4 array element as one 12-byte load (the w of a neighbour
// is not used by the pair terms).
__device__ __forceinline__ float3 ld_xyz(const float4* p) {
    const float* f = reinterpret_cast<const float*>(p);
    return make_float3(f[0], f[1], f[2]);
}

// LDS staging of neighbour rows, per wavefront: the wavefront loads each
// stencil row's run once, coalesced, into its own LDS slice and the lanes
// read their candidates from there instead of gathering them from memory,
// where the lanes of a row touch the same particles many times.  The density
// pass stages positions, kStagePos at a time, the force pass neighbour
// records (two float4), kStageRecs at a time; a run is about 80 to 100
// particles, more only where few particles of a wavefront lie in each cell
// beside full ones, as in the outermost layer of a fluid.
constexpr uint32_t kStagePos = 252;
constexpr uint32_t kStageRecs = 160;  // 5 KB a wavefront: 32 wavefronts in a CU's LDS

// The cells of a wavefront's particles (the lanes are consecutive sorted
// particles, so about eight to twelve distinct ones in the bulk of a fluid
// and up to 64 at its edges), and what each of the nine stencil rows holds
// around them.  Entry (row, c) is the first sorted index B0 of cells
// cx-1..cx+1 of the row at the c-th cell, from the row's run's first (11
// bits), and, in 7 bits each, the distances from B0 to the end of cell cx-1,
// the start of cell cx+1 and the end of cell cx+1 (0 in the last: the row is
// empty there).
struct WaveCells {
    uint32_t row[9][64];
    uint32_t key[64];       // a cell's key
    uint32_t lo[9], hi[9];  // the rows' runs
    uint32_t most[9];       // most particles in three cells
    uint8_t sides[64];      // kSide* of the grid around a cell
};
constexpr uint32_t kWaveCellsTemp = 9 * 64;  // words that wave_cells needs besides
constexpr uint32_t kSideLowY = 1u, kSideHighY = 2u, kSideLowZ = 4u, kSideHighZ = 8u, kSideLeft = 16u,
                   kSideRight = 32u;

// A wavefront's slice in the density pass: the positions of the current run
// as (x, y) pairs and z (the lanes of one cell read the same candidate and
// those of the next cell one about eight further: 8- and 4-byte reads of
// such addresses are free of bank conflicts, where 12- and 16-byte reads of
// whole positions cost 1.5 times as much per candidate, the test and the sum
// included: 33 against 21 SIMD cycles).
struct DensityStage {
    float2 xy[kStagePos + 4];
    float z[kStagePos + 4];
    WaveCells cells;
    __device__ __forceinline__ uint32_t* temp() { return reinterpret_cast<uint32_t*>(xy); }
};
static_assert(offsetof(DensityStage, cells) >= sizeof(uint32_t) * kWaveCellsTemp, "wave_cells' temporary words");

// The runs of a wavefront's nine rows: row r's first index and length word
// (as in the runs table), in lane r.
struct WaveRuns {
    uint32_t lo = 0u, info = 0u;
    __device__ __forceinline__ uint32_t first(int row) const {
        return (uint32_t)__builtin_amdgcn_readlane((int)lo, row);
    }
    __device__ __forceinline__ uint32_t word(int row) const {
        return (uint32_t)__builtin_amdgcn_readlane((int)info, row);
    }
};

// Fills wc for the wavefront (every lane calls it) and gives each lane the
// index of its cell there, and the wavefront its runs: row r's run goes from
// the smallest B0 to the largest end of the row's entries.  A row in which
// three cells hold more than 127 particles has kRunLookup set, its lanes look
// their ranges up (other_row); one whose run is too long has kRunFar set and no
// length, and is read from memory.  (1,048,576 particles on cells of 2 h, where
// one such cell used to send all nine rows of its wavefront to memory: density
// 580 us so and 330 now, forces 1,190 and 670; on cells of 1.3 h, where some
// rows are longer than a mask, forces 271 and 157.)
// `temp`: nine times 64 words of LDS, `stride` words apart, free again afterwards.
//
// The nine rows of the cells are looked up by (cell, row) pairs, a pair a
// lane and two a round: one round of twelve loads for the 64 particles in the
// bulk of a fluid, where every lane looking up its own nine rows takes 54
// loads of addresses that mostly coincide.
__device__ __forceinline__ void wave_cells(WaveCells& wc, uint32_t* __restrict__ temp, uint32_t stride, const RowWalker& w,
                                           const fg_common_fluid_params& cp, uint32_t key_base,
                                           const uint32_t* __restrict__ start, const uint32_t* __restrict__ end,
                                           uint32_t n, uint32_t& cell, WaveRuns& runs) {
    const uint32_t lane = __lane_id();
    const uint32_t key = key_base + linear_key(w.cx, w.cy, w.cz, cp);
    const uint32_t before = (uint32_t)__shfl_up((int)key, 1);
    const bool head = lane == 0u || key != before;
    const uint64_t heads = __ballot(head);
    const uint32_t pairs = 9u * (uint32_t)__popcll(heads);
    cell = __builtin_amdgcn_mbcnt_hi((uint32_t)(heads >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)heads, 0u)) -
           (head ? 0u : 1u);
    if (head) {
        wc.key[cell] = key;
        wc.sides[cell] = (uint8_t)((w.cy > 0 ? kSideLowY : 0u) | (w.cy + 1 < cp.bucket_size.y ? kSideHighY : 0u) |
                         (w.cz > 0 ? kSideLowZ : 0u) | (w.cz + 1 < cp.bucket_size.z ? kSideHighZ : 0u) |
                         (w.cx > 0 ? kSideLeft : 0u) | (w.cx + 1 < cp.bucket_size.x ? kSideRight : 0u));
    }
    if (lane < 9u) {
        wc.lo[lane] = kEmpty;
        wc.hi[lane] = wc.most[lane] = 0u;
    }
    wave_lds_sync();
    const uint32_t by = (uint32_t)cp.bucket_size.x, bz = by * (uint32_t)cp.bucket_size.y;
    for (uint32_t q0 = lane; q0 < pairs; q0 += 128u) {
        uint32_t s[2][3], e[2][3];
        bool valid[2];
#pragma unroll
        for (uint32_t u = 0; u < 2u; u++) {
            const uint32_t q = q0 + 64u * u < pairs ? q0 + 64u * u : q0;  // (the second may be the first again)
            const uint32_t c = q / 9u, row = q - 9u * c, z3 = row / 3u, y3 = row - 3u * z3;  // dy + 1, dz + 1
            const uint32_t k = wc.key[c], sides = wc.sides[c];
            const uint32_t need = (y3 == 0u ? kSideLowY : 0u) | (y3 == 2u ? kSideHighY : 0u) |
                                  (z3 == 0u ? kSideLowZ : 0u) | (z3 == 2u ? kSideHighZ : 0u);
            const bool left = (sides & kSideLeft) != 0u, right = (sides & kSideRight) != 0u;
            valid[u] = (sides & need) == need;
            // (a row outside the grid reads the cell's own)
            const uint32_t m = valid[u] ? k + y3 * by + z3 * bz - (by + bz) : k;
            const uint32_t l = left ? m - 1u : m, r = right ? m + 1u : m;
            s[u][0] = start[l];
            s[u][1] = start[m];
            s[u][2] = start[r];
            e[u][0] = end[l];
            e[u][1] = end[m];
            e[u][2] = end[r];
            if (!left) s[u][0] = kEmpty;
            if (!right) s[u][2] = kEmpty;
        }
#pragma unroll
        for (uint32_t u = 0; u < 2u; u++) {
            const uint32_t q = q0 + 64u * u < pairs ? q0 + 64u * u : q0;
            const uint32_t c = q / 9u, row = q - 9u * c;
            // an empty cell's start is the largest value, its end is stale
            const uint32_t e0 = s[u][0] != kEmpty ? min(e[u][0], n) : 0u, e1 = s[u][1] != kEmpty ? min(e[u][1], n) : 0u;
            const uint32_t e2 = s[u][2] != kEmpty ? min(e[u][2], n) : 0u;
            const uint32_t b0 = min(min(s[u][0], s[u][1]), s[u][2]), b3 = max(max(e0, e1), e2);
            uint32_t d = 0u;
            if (valid[u] && b0 < b3) {
                const uint32_t d1 = s[u][0] != kEmpty ? e0 - b0 : 0u, d2 = s[u][2] != kEmpty ? s[u][2] - b0 : b3 - b0;
                atomicMax(&wc.most[row], b3 - b0);
                d = ((d1 & 127u) << 11) | ((d2 & 127u) << 18) | ((b3 - b0) << 25);
                atomicMin(&wc.lo[row], b0);
                atomicMax(&wc.hi[row], b3);
            }
            wc.row[row][c] = b0;
            temp[stride * row + c] = d;
        }
    }
    wave_lds_sync();
    for (uint32_t q = lane; q < pairs; q += 64u) {  // the first indices from the runs' firsts
        const uint32_t c = q / 9u, row = q - 9u * c, d = temp[stride * row + c];
        wc.row[row][c] = d ? ((wc.row[row][c] - wc.lo[row]) & kRunMax) | d : 0u;
    }
    if (lane < 9u && wc.hi[lane] != 0u) {
        runs.lo = wc.lo[lane];
        const uint32_t len = wc.hi[lane] - runs.lo, most = wc.most[lane];
        runs.info = len > kRunMax || (len > kRunSparse && len > kRunSpread * most) ? kRunFar
                                                                           : len | (most > 127u ? kRunLookup : 0u);
    }
    wave_lds_sync();
}

// A lane's range in a row, from its run's first index: the row's cells after
// culling by distance (row_keys).
struct LaneRow {
    uint32_t off, len;  // len 0: no candidates
};
__device__ __forceinline__ LaneRow lane_row(const WaveCells& wc, int row, uint32_t cell, bool active,
                                            const RowWalker& w, float cut) {
    const int dz = row / 3 - 1, dy = row % 3 - 1;
    const float gy = dy < 0 ? w.gy_lo : (dy > 0 ? w.gy_hi : 0.0f);
    const float gz = dz < 0 ? w.gz_lo : (dz > 0 ? w.gz_hi : 0.0f);
    const float gyz = gy + gz;
    const uint32_t c = wc.row[row][cell];
    const uint32_t first = gyz + w.gx_lo < cut ? 0u : (c >> 11) & 127u;
    const uint32_t last = gyz + w.gx_hi < cut ? c >> 25 : (c >> 18) & 127u;
    return LaneRow{(c & kRunMax) + first, active && gyz < cut && last > first ? last - first : 0u};
}

// lane_row of a row that WaveCells does not hold: the range from the cell
// tables (off is of use within kRunMax only).
__device__ __forceinline__ LaneRow other_row(int row, bool active, const float4& p, uint32_t lo, float cut,
                                             const fg_common_fluid_params& cp, uint32_t key_base,
                                             const uint32_t* __restrict__ start, const uint32_t* __restrict__ end,
                                             uint32_t n) {
    uint32_t rb = lo, re = lo;
    const bool has = active && row_range(make_rows(p, cp), row % 3 - 1, row / 3 - 1, cut, cp, key_base, start, end, n,
                                         rb, re);
    return LaneRow{rb - lo, has ? re - rb : 0u};
}

// A run's length word, from its word of wave_cells and the lanes' candidates in it.
__device__ __forceinline__ uint32_t run_word(uint32_t word, uint32_t len) {
    word &= kRunLength | kRunFar;
    if (__ballot(len > 32u) != 0ull) word |= kRunWide;
    if (__ballot(len > kRowMaskBits) != 0ull) word |= kRunLong;
    return word;
}

// Wavefront w's runs (first index and word of each row), for the force pass.
__device__ __forceinline__ void store_runs(const WaveRuns& runs, uint32_t w, unsigned long long* masks, uint32_t n) {
    if (__lane_id() < 9u) {
        uint32_t* t = nbr_runs(masks, n) + (size_t)kRunWords * w + __lane_id();
        t[0] = runs.lo;
        t[9] = runs.info;
    }
}

// Poly6 sum over four candidates; bit u of the returned nibble is set when
// candidate u lies within h.
//
// The fused multiply-adds are written out (and contraction is off here), so
// every schedule and workgroup size that inlines this evaluates exactly the
// same operations.
#pragma clang fp contract(off)
__device__ __forceinline__ uint32_t density4(const float4& p, const float3& q0, const float3& q1, const float3& q2,
                                             const float3& q3, float h2u, float hhu, float& acc) {
    const float3 q[4] = {q0, q1, q2, q3};
    uint32_t nib = 0;
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const float dx = p.x - q[u].x, dy = p.y - q[u].y, dz = p.z - q[u].z;
        const float r2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
        const float t = h2u - r2;
        const bool hit = r2 < hhu;
        acc = hit ? __builtin_fmaf(t * t, t, acc) : acc;
        nib |= hit ? (1u << u) : 0u;
    }
    return nib;
}
#pragma clang fp contract(fast)

// rho_p[i] = (max(1, rho), k (rho - rho0)) (K_FluidSim.cu:246-249) and, when
// rec is given, particle i's neighbour record from its sorted position p,
// sorted velocity v and (1/rho_p.x, rho_p.y/rho_p.x).
#pragma clang fp contract(off)
__device__ __forceinline__ void store_record(uint32_t i, float2 rp, const float4& p, const float4& v,
                                             float4* __restrict__ rec) {
    const float a = 1.0f / rp.x;
    rec[2 * (size_t)i] = make_float4(p.x, p.y, p.z, a);
    rec[2 * (size_t)i + 1] = make_float4(v.x, v.y, v.z, rp.y * a);
}
__device__ __forceinline__ void store_density(uint32_t i, float rho, float k, float rho0, float2* __restrict__ rho_p,
                                              float4* __restrict__ rec, const float4& p, const float4& v) {
    const float2 rp = make_float2(fmaxf(1.0f, rho), k * (rho - rho0));
    rho_p[i] = rp;
    if (rec) store_record(i, rp, p, v, rec);
}
#pragma clang fp contract(fast)

// One stencil row of the density pass: the len candidates pp[0, len) of the
// sorted positions, in groups of four in sorted order (a short last group
// padded with far points) added to acc, and the row's mask (0 for rows
// longer than 64 candidates, which are never read through their mask).
template <bool MASKS>
__device__ __forceinline__ unsigned long long density_row(const float4& p, const float4* __restrict__ pp,
                                                          uint32_t len, float h2u, float hhu, float& acc) {
    unsigned long long msk = 0ull;
    const uint32_t n4 = len & ~3u;
    uint32_t kk = 0;
    if (n4) {
        // Software-pipelined groups of four: the next group's loads are
        // in flight while the current group is evaluated.
        float3 a0 = ld_xyz(pp), a1 = ld_xyz(pp + 1), a2 = ld_xyz(pp + 2), a3 = ld_xyz(pp + 3);
        for (; kk + 4 < n4; kk += 4) {
            pp += 4;
            const float3 b0 = ld_xyz(pp), b1 = ld_xyz(pp + 1), b2 = ld_xyz(pp + 2), b3 = ld_xyz(pp + 3);
            const uint32_t nib = density4(p, a0, a1, a2, a3, h2u, hhu, acc);
            if (MASKS) msk |= (unsigned long long)nib << (kk & 63u);
            a0 = b0; a1 = b1; a2 = b2; a3 = b3;
        }
        const uint32_t nib = density4(p, a0, a1, a2, a3, h2u, hhu, acc);
        if (MASKS) msk |= (unsigned long long)nib << (kk & 63u);
        kk += 4;
        pp += 4;
    }
    if (kk < len) {  // 1-3 remaining candidates; the others are masked out
        const uint32_t rest = len - kk;
        const float3 far = make_float3(3.0e38f, 3.0e38f, 3.0e38f);
        const float3 t0 = ld_xyz(pp);
        const float3 t1 = rest > 1 ? ld_xyz(pp + 1) : far;
        const float3 t2 = rest > 2 ? ld_xyz(pp + 2) : far;
        const uint32_t nib = density4(p, t0, t1, t2, far, h2u, hhu, acc);
        if (MASKS) msk |= (unsigned long long)nib << (kk & 63u);
    }
    return len <= kRowMaskBits ? msk : 0ull;
}

// density4 on four candidates of the staged run, with the same operations, a
// miss adding +0 (acc starts at +0 and never becomes -0, so that changes no
// bit), and the hit bits shifted into `bits` from below, the first candidate
// first.  Candidates from `rest` on are no hits.
//
// SAME: h2u and hhu are the same value (always so at simulation scale 1), and
// no r2 is NaN (stage_number).  Then h2u - r2 is positive exactly
// for the hits, the sum takes its positive part, and the hit bit is the sign
// of r2 - hhu: 11 instructions a candidate.
// Otherwise the compares, selects and shifts are written out: as selects of 0
// and 1 the mask would cost two instructions a candidate more.  A compare's
// result is read three instructions after it at the earliest (two must lie
// between).
#pragma clang fp contract(off)
template <bool SAME, bool ALL>
__device__ __forceinline__ void density_group(const float4& p, const float2* __restrict__ xy,
                                              const float* __restrict__ z, uint32_t rest, float h2u, float hhu,
                                              float& acc, uint32_t& bits) {
    float r2[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const float dx = p.x - xy[u].x, dy = p.y - xy[u].y, dz = p.z - z[u];
        r2[u] = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
    }
    if constexpr (SAME) {
#pragma unroll
        for (uint32_t u = 0; u < 4u; u++) {
            float d = r2[u] - hhu;
            if (!ALL && u > 0u) d = u < rest ? d : 1.0f;
            bits = __builtin_amdgcn_alignbit(bits, __float_as_uint(d), 31);
            const float t = __builtin_fmaxf(-d, 0.0f);
            acc = __builtin_fmaf(t * t, t, acc);
        }
        return;
    }
    float t[4];
#pragma unroll
    for (int u = 0; u < 4; u++) t[u] = h2u - r2[u];
    const float l1 = ALL || rest > 1u ? hhu : -1.0f, l2 = ALL || rest > 2u ? hhu : -1.0f;
    const float l3 = ALL ? hhu : -1.0f;
    uint64_t c0, c1, c2, c3;
    asm("v_cmp_lt_f32_e64 %[c0], %[a0], %[m0]\n\t"
        "v_cmp_lt_f32_e64 %[c1], %[a1], %[m1]\n\t"
        "v_cmp_lt_f32_e64 %[c2], %[a2], %[m2]\n\t"
        "v_cmp_lt_f32_e64 %[c3], %[a3], %[m3]\n\t"
        "v_cndmask_b32_e64 %[t0], 0, %[t0], %[c0]\n\t"
        "v_addc_co_u32_e64 %[b], vcc, %[b], %[b], %[c0]\n\t"
        "v_cndmask_b32_e64 %[t1], 0, %[t1], %[c1]\n\t"
        "v_addc_co_u32_e64 %[b], vcc, %[b], %[b], %[c1]\n\t"
        "v_cndmask_b32_e64 %[t2], 0, %[t2], %[c2]\n\t"
        "v_addc_co_u32_e64 %[b], vcc, %[b], %[b], %[c2]\n\t"
        "v_cndmask_b32_e64 %[t3], 0, %[t3], %[c3]\n\t"
        "v_addc_co_u32_e64 %[b], vcc, %[b], %[b], %[c3]"
        : [c0] "=&s"(c0), [c1] "=&s"(c1), [c2] "=&s"(c2), [c3] "=&s"(c3), [t0] "+&v"(t[0]), [t1] "+&v"(t[1]),
          [t2] "+&v"(t[2]), [t3] "+&v"(t[3]), [b] "+&v"(bits)
        : [a0] "v"(r2[0]), [a1] "v"(r2[1]), [a2] "v"(r2[2]), [a3] "v"(r2[3]), [m0] "v"(hhu), [m1] "v"(l1),
          [m2] "v"(l2), [m3] "v"(l3)
        : "vcc");
#pragma unroll
    for (int u = 0; u < 4; u++) acc = __builtin_fmaf(t[u] * t[u], t[u], acc);
}
#pragma clang fp contract(fast)

// A coordinate as it is staged: a NaN becomes an infinity.  A particle whose
// own position is finite (the others have no hits, and walk nothing) then gets
// an infinite r2 from one that is not, never a NaN, and no hit.  (Written out:
// of the builtin with these bounds the compiler makes two instructions, 1% of
// the density pass.  A median of a NaN is the minimum of the other two, or of a
// signalling one the last.)
__device__ __forceinline__ float stage_number(float v) {
    float r = v;
    asm("v_med3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "s"(-__builtin_inff()), "v"(__builtin_inff()));
    return r;
}
__device__ __forceinline__ bool finite_position(const float4& p) {
    return fabsf(p.x) < __builtin_inff() && fabsf(p.y) < __builtin_inff() && fabsf(p.z) < __builtin_inff();
}

// Part of a stencil row of the density pass from the staged run: cnt
// candidates from slice index `at`, the first one bit `bit` of the row's mask.
template <bool MASKS, bool SAME>
__device__ __forceinline__ void density_row_staged(const float4& p, const DensityStage& st, uint32_t at, uint32_t cnt,
                                                   uint32_t bit, float h2u, float hhu, float& acc,
                                                   unsigned long long& mask) {
    for (;;) {  // a row rarely has more than 32 candidates
        const uint32_t c = min(cnt, 32u);
        const float2* xy = st.xy + at;
        const float* z = st.z + at;
        uint32_t bits = 0u, k = 0u;
        for (; k + 4u <= c; k += 4u) density_group<SAME, true>(p, xy + k, z + k, 4u, h2u, hhu, acc, bits);
        if (k < c) {  // up to three more; what lies past them in the slice is no hit
            density_group<SAME, false>(p, xy + k, z + k, c - k, h2u, hhu, acc, bits);
            k += 4u;
        }
        // candidate j was shifted in as bit k - 1 - j
        if (MASKS) mask |= (unsigned long long)(__builtin_bitreverse32(bits) >> (32u - k)) << (bit & 63u);
        if (cnt <= 32u) break;
        cnt -= 32u;
        at += 32u;
        bit += 32u;
    }
}

// The row loop of the density pass for a whole wavefront (every lane present;
// a lane of an inactive particle, or one past the last particle, takes part
// with no rows and writes no masks): each row's run staged in the wavefront's
// LDS slice, the next row's positions loaded into registers while this row
// is walked.  Same candidates, same order, same sums and masks as the row
// loop of density_particle.
//
// Bound by VALU issue: 4,724 instructions a wavefront, 3,800 of them in the
// walks (65 groups of four candidates, which its longest lane per row sets);
// 30% of a wavefront's time is waiting.  8,388,608 particles take 0.83 ms
// against 0.87 with per-lane lookups row by row and whole positions in LDS,
// 1,048,576 at the start of a dam break 99.8 us against 98.5, and on cells of
// 2 h 330 against 467.
template <bool MASKS>
__device__ __forceinline__ float density_rows_staged(uint32_t i, bool active, const float4& p,
                                                    const float4* __restrict__ sp,
                                                    const uint32_t* __restrict__ start,
                                                    const uint32_t* __restrict__ end, uint32_t n,
                                                    const fg_common_fluid_params& cp, uint32_t key_base,
                                                    unsigned long long* __restrict__ masks, DensityStage& st) {
    const float s = cp.simulation_scale, s2 = s * s;
    const float h = cp.kernel_radius, hh = h * h;
    const float hu = h / s, hhu = hu * hu, h2u = cp.kernel_radius_squared / s2;
    const float cut = hh * 1.0001f;
    const uint32_t lane = __lane_id();
    const uint32_t wave = __builtin_amdgcn_readfirstlane(i >> 6);
    const bool table = MASKS && n >= kRunMinParticles;
    const RowWalker w = make_rows(p, cp);
    uint32_t cell;
    WaveRuns runs;
    wave_cells(st.cells, st.temp(), 64u, w, cp, key_base, start, end, n, cell, runs);
    const bool same = __builtin_amdgcn_readfirstlane(__float_as_uint(h2u) == __float_as_uint(hhu) ? 1u : 0u) != 0u;
    const bool walks = active && finite_position(p);
    uint16_t* offs = MASKS ? nbr_offs(masks, n) + (size_t)9 * 64 * wave + lane : nullptr;
    uint32_t words = 0u;
    unsigned long long msk = 0ull, last = 0ull;
    float acc = 0.0f;
    float3 n0 = make_float3(0.0f, 0.0f, 0.0f), n1 = n0;
    auto fetch = [&](int row) {
        const uint32_t len = runs.word(row) & kRunLength;
        const float4* q = sp + runs.first(row) + lane;
        if (lane < len) n0 = ld_xyz(q);
        if (lane + 64u < len) n1 = ld_xyz(q + 64);
    };
    auto put = [&](uint32_t k, const float3& q) {
        st.xy[k] = make_float2(stage_number(q.x), stage_number(q.y));
        st.z[k] = stage_number(q.z);
    };
    fetch(0);
    for (int row = 0; row < 9; row++) {
        const uint32_t info = runs.word(row), len = info & kRunLength, lo = runs.first(row);  // the same on every lane
        LaneRow r = lane_row(st.cells, row, cell, walks, w, cut);
        if (info & (kRunLookup | kRunFar)) r = other_row(row, walks, p, lo, cut, cp, key_base, start, end, n);
        if (table) {
            const uint32_t word = run_word(info, r.len);
            words = (int)lane == row ? word : words;
        }
        msk = 0ull;
        const bool whole = r.len <= kRowMaskBits;
        if (info & kRunFar) {
            if (r.len) msk = density_row<MASKS>(p, sp + lo + r.off, r.len, h2u, hhu, acc);
            r.len = 0u;
        }
        // the lane's candidates among the staged positions [at, at + kStagePos) of the run
        auto walk = [&](uint32_t at) {
            const uint32_t a = max(r.off, at), b = min(r.off + r.len, at + kStagePos);
            if (a < b) {
                if (same) density_row_staged<MASKS, true>(p, st, a - at, b - a, a - r.off, h2u, hhu, acc, msk);
                else density_row_staged<MASKS, false>(p, st, a - at, b - a, a - r.off, h2u, hhu, acc, msk);
            }
        };
        for (uint32_t at = 0u;;) {  // (a run rarely fills the slice)
            const uint32_t cnt = min(len - at, kStagePos);
            if (at == 0u) {
                if (lane < cnt) put(lane, n0);
                if (lane + 64u < cnt) put(lane + 64u, n1);
                // The last row's mask and this row's offsets are stored
                // before the next row's loads are issued: loads and stores
                // are waited for together, and a store issued after the
                // walk would hold up the next row's positions.
                if (MASKS && active && row > 0) masks[(size_t)(row - 1) * n + i] = last;
                if (table) offs[64 * row] = (uint16_t)r.off;
                if (row < 8) fetch(row + 1);
            }
            for (uint32_t k = lane + (at == 0u ? 128u : 0u); k < cnt; k += 64u) put(k, ld_xyz(sp + lo + at + k));
            wave_lds_sync();
            walk(at);
            wave_lds_sync();  // every lane's reads before the next stores
            at += kStagePos;
            if (at >= len) break;
        }
        last = whole ? msk : 0ull;
    }
    if (MASKS && active) masks[(size_t)8 * n + i] = last;
    if (table) {
        runs.info = words;
        store_runs(runs, wave, masks, n);
    }
    return acc;
}

// A wavefront's LDS in the flat density schedule: what finding its rows takes,
// then each lane's table of them, 5 KB together (32 wavefronts in a CU's LDS).
union FlatWave {
    struct {
        WaveCells cells;
        uint32_t temp[kWaveCellsTemp];
    } find;
    uint32_t rows[2][9][64];
};
static_assert(sizeof(FlatWave) <= 5120, "32 wavefronts in 160 KB");

// The flat schedule's per-lane table: first and one-past-last sorted index of
// each of the 9 rows (equal for a culled row).  `one_grid`: the lanes of a full
// wavefront here hold particles of one grid.
struct FlatRanges {
    FlatWave* wave;
    bool one_grid;
    __device__ __forceinline__ uint32_t& b(int r) const { return wave->rows[0][r][__lane_id()]; }
    __device__ __forceinline__ uint32_t& e(int r) const { return wave->rows[1][r][__lane_id()]; }
};

// Fills the table of a whole wavefront of one grid, its rows found together
// (wave_cells), and, with `masks`, the runs' table of wavefront `wave`.
// Density of 1,048,576 and 100,920 particles 244 and 44.1 us where every lane
// looked up its own rows besides, 237 and 39.4 us so (235 and 38.4 without the
// runs, 228 and 39.9 with the lanes' own lookups and no runs: the table is
// always left, so that a force pass may walk rows after it).
__device__ __forceinline__ void flat_rows(const FlatRanges& flat, bool active, const float4& p,
                                          const fg_common_fluid_params& cp, uint32_t key_base,
                                          const uint32_t* __restrict__ start, const uint32_t* __restrict__ end,
                                          uint32_t n, uint32_t wave, unsigned long long* __restrict__ masks) {
    const float cut = cp.kernel_radius * cp.kernel_radius * 1.0001f;
    const RowWalker w = make_rows(p, cp);
    WaveCells& cells = flat.wave->find.cells;
    uint32_t cell;
    WaveRuns runs;
    wave_cells(cells, flat.wave->find.temp, 64u, w, cp, key_base, start, end, n, cell, runs);
    uint32_t found[9];
#pragma unroll
    for (int row = 0; row < 9; row++) {
        const LaneRow r = lane_row(cells, row, cell, active, w, cut);
        found[row] = r.off | r.len << 16;
    }
    wave_lds_sync();  // every lane's reads before the table
#pragma unroll
    for (int row = 0; row < 9; row++) {
        flat.b(row) = runs.first(row) + (found[row] & 0xFFFFu);
        flat.e(row) = flat.b(row) + (found[row] >> 16);
    }
    uint16_t* offs = nbr_offs(masks, n) + (size_t)9 * 64 * wave + __lane_id();
    uint32_t words = 0u;
#pragma unroll 1
    for (int row = 0; row < 9; row++) {
        const uint32_t info = runs.word(row), lo = runs.first(row);
        if (info & (kRunLookup | kRunFar)) {
            const LaneRow r = other_row(row, active, p, lo, cut, cp, key_base, start, end, n);
            flat.b(row) = lo + r.off;
            flat.e(row) = lo + r.off + r.len;
        }
        if (masks) {
            offs[64 * row] = (uint16_t)(flat.b(row) - lo);
            const uint32_t word = run_word(info, flat.e(row) - flat.b(row));
            words = (int)__lane_id() == row ? word : words;
        }
    }
    runs.info = words;
    if (masks) store_runs(runs, wave, masks, n);
}

// Density of sorted particle i (i < n): rho_p[i] = (max(1, rho), k (rho - rho0)),
// and, with MASKS, its row masks and its neighbour record (sv, the sorted
// velocities, is read only then).
//
// Two schedules give bit-identical sums (rows in order, candidates of a row
// in groups of four in sorted order, a short last group padded with far
// points): the row loop, where a wavefront waits at every row for its lane
// with the longest row, and the flat schedule (with a row table), where each
// lane walks its own candidate stream across rows.  Given an LDS slice
// (`stage`) and a whole wavefront, the row loop reads each row's candidates
// from LDS (density_rows_staged).  A whole wavefront may call it with
// i >= n on its last lanes, which then only take part.
template <bool MASKS>
__device__ __forceinline__ void density_particle(uint32_t i, const float4* __restrict__ sp,
                                                 const float4* __restrict__ sv, float2* __restrict__ rho_p, const uint32_t* __restrict__ start,
                                                 const uint32_t* __restrict__ end, uint32_t n, float k, float rho0,
                                                 float m, const fg_common_fluid_params& cp,
                                                 const fg_kernels_cache& kc, uint32_t key_base,
                                                 unsigned long long* __restrict__ masks,
                                                 const FlatRanges* flat = nullptr, DensityStage* stage = nullptr) {
    const bool valid = i < n;
    const float4 p = sp[min(i, n - 1u)];
    float4* rec = MASKS ? nbr_records(masks, n) : nullptr;
    // The staged row loop needs every lane of the wavefront (a row's run is
    // its lanes' together); otherwise the rows are read from memory.
    const bool whole = __ballot(1) == ~0ull;
    if (stage != nullptr && flat == nullptr && whole) {
        const float sum =
            density_rows_staged<MASKS>(i, valid && p.w > 0.0f, p, sp, start, end, n, cp, key_base, masks, *stage);
        if (!valid) return;
        const float4 v = MASKS ? sv[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (p.w > 0.0f) {
            const float s2 = cp.simulation_scale * cp.simulation_scale;
            store_density(i, m * kc.kPoly6 * (s2 * s2 * s2) * sum, k, rho0, rho_p, rec, p, v);
        } else if (MASKS) {
            store_record(i, rho_p[i], p, v, rec);
        }
        return;
    }
    const bool together = flat && flat->one_grid && whole;
    if (together)
        flat_rows(*flat, valid && p.w > 0.0f, p, cp, key_base, start, end, n, __builtin_amdgcn_readfirstlane(i >> 6),
                  MASKS && n >= kRunMinParticles ? masks : nullptr);
    if (!valid) return;
    const float4 v = MASKS ? sv[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (!(p.w > 0.0f)) {
        // (rho, p) is left as it is; neighbours still read it
        if (MASKS) store_record(i, rho_p[i], p, v, rec);
        return;
    }
    // Distances are compared unscaled: r_u = r / s, so r < h <=> r_u^2 < (h/s)^2
    // and h^2 - r^2 = s^2 (h^2/s^2 - r_u^2).
    const float s = cp.simulation_scale, s2 = s * s;
    const float h = cp.kernel_radius, hh = h * h;
    const float hu = h / s, hhu = hu * hu, h2u = cp.kernel_radius_squared / s2;
    const float cut = hh * 1.0001f;
    const RowWalker w = make_rows(p, cp);
    float acc = 0.0f;
    if (flat) {
        if (!together) {
#pragma unroll
            for (int row = 0; row < 9; row++) {
                uint32_t rb = 0, re = 0;
                if (!row_range(w, row % 3 - 1, row / 3 - 1, cut, cp, key_base, start, end, n, rb, re)) rb = re = 0;
                flat->b(row) = rb;
                flat->e(row) = re;
            }
        }
        const float3 far = make_float3(3.0e38f, 3.0e38f, 3.0e38f);
        int row = -1;
        uint32_t j = 0, rb = 0, re = 0;
        unsigned long long msk = 0ull;
        for (;;) {
            while (j >= re) {
                if (MASKS && row >= 0) masks[(size_t)row * n + i] = msk;
                if (row == 8) break;
                row++;
                rb = flat->b(row);
                re = flat->e(row);
                j = rb;
                msk = 0ull;
            }
            if (j >= re) break;
            const uint32_t rest = re - j;
            const float4* pp = sp + j;
            const float3 t0 = ld_xyz(pp);
            const float3 t1 = rest > 1 ? ld_xyz(pp + 1) : far;
            const float3 t2 = rest > 2 ? ld_xyz(pp + 2) : far;
            const float3 t3 = rest > 3 ? ld_xyz(pp + 3) : far;
            const uint32_t nib = density4(p, t0, t1, t2, t3, h2u, hhu, acc);
            if (MASKS) msk |= (unsigned long long)nib << ((j - rb) & 63u);
            j += 4;
        }
        store_density(i, m * kc.kPoly6 * (s2 * s2 * s2) * acc, k, rho0, rho_p, rec, p, v);
        return;
    }
    for (int row = 0; row < 9; row++) {
        const int dz = row / 3 - 1, dy = row % 3 - 1;
        unsigned long long msk = 0ull;
        uint32_t rb, re;
        if (row_range(w, dy, dz, cut, cp, key_base, start, end, n, rb, re))
            msk = density_row<MASKS>(p, sp + rb, re - rb, h2u, hhu, acc);
        if (MASKS) masks[(size_t)row * n + i] = msk;
    }
    store_density(i, m * kc.kPoly6 * (s2 * s2 * s2) * acc, k, rho0, rho_p, rec, p, v);
}

// Pressure and viscosity terms of one neighbour j (r < h checked again, so
// the same code serves rows without a mask), from aj = 1/rho_j and
// bj = p_j/rho_j: (p_i + p_j)/rho_j = p_i aj + bj.
struct PairAcc {
    float px, py, pz, vx, vy, vz;
};

#pragma clang fp contract(off)
// The accumulation of one pair with r2u = |x_i - x_j|^2 (unscaled) < h^2.
__device__ __forceinline__ void pair_accumulate(PairAcc& A, float dx, float dy, float dz, float r2u,
                                                const float4& vel, float pri, float3 vj, float aj, float bj,
                                                float h, float s) {
    const float iru = __builtin_amdgcn_rsqf(r2u);
    const float hr = __builtin_fmaf(-(r2u * iru), s, h);
    const float cp_ = hr * hr * __builtin_fmaf(pri, aj, bj) * iru;
    A.px = __builtin_fmaf(dx, cp_, A.px);
    A.py = __builtin_fmaf(dy, cp_, A.py);
    A.pz = __builtin_fmaf(dz, cp_, A.pz);
    const float cv = hr * aj;
    A.vx = __builtin_fmaf(vj.x - vel.x, cv, A.vx);
    A.vy = __builtin_fmaf(vj.y - vel.y, cv, A.vy);
    A.vz = __builtin_fmaf(vj.z - vel.z, cv, A.vz);
}

__device__ __forceinline__ void pair_term(PairAcc& A, uint32_t i, uint32_t j, const float4& pos, const float4& vel,
                                          float pri, float3 q, float3 vj, float aj, float bj, float h, float s,
                                          float hhu) {
    const float dx = pos.x - q.x, dy = pos.y - q.y, dz = pos.z - q.z;
    const float r2u = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));  // unscaled
    if (r2u < hhu && j != i) pair_accumulate(A, dx, dy, dz, r2u, vel, pri, vj, aj, bj, h, s);
}

// A pair from a neighbour mask (self bit cleared).  The density pass set the
// bit after the same test on the same r2u (the same operations on the same
// sorted positions), so r2u < h^2 holds and is not tested again: without
// the branch the neighbour's velocity and inverse-density loads are issued
// together with its position load instead of after the test.
__device__ __forceinline__ void pair_term_masked(PairAcc& A, const float4& pos, const float4& vel, float pri,
                                                 float3 q, float3 vj, float aj, float bj, float h, float s) {
    const float dx = pos.x - q.x, dy = pos.y - q.y, dz = pos.z - q.z;
    const float r2u = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
    pair_accumulate(A, dx, dy, dz, r2u, vel, pri, vj, aj, bj, h, s);
}

// The same from a stored (rho_j, p_j) (rows without a mask), with the
// (1/rho_j, p_j/rho_j) the density pass stores beside the masks.
__device__ __forceinline__ void pair_term_rp(PairAcc& A, uint32_t i, uint32_t j, const float4& pos,
                                             const float4& vel, float pri, float3 q, float3 vj, float2 dpj, float h,
                                             float s, float hhu) {
    const float aj = 1.0f / dpj.x;
    pair_term(A, i, j, pos, vel, pri, q, vj, aj, dpj.y * aj, h, s, hhu);
}
#pragma clang fp contract(fast)

// The neighbours of one row from its mask mm (self bit cleared), bit k
// being record first + k, in ascending order, two per iteration.  Record j
// is (rec[2 j], rec[2 j + 1]), in memory.
// The mask is walked as two 32-bit words, low word first (the same
// ascending order): 32-bit bit scans and clears, and rows of at most 32
// candidates never enter the second loop.
__device__ __forceinline__ void walk_row_mask(PairAcc& A, unsigned long long mm, uint32_t first,
                                              const float4* __restrict__ rec, const float4& pos, const float4& vel,
                                              float pri, float h, float s) {
    uint32_t word = (uint32_t)mm, base = first;
    for (int half = 0; half < 2; half++) {
        while (word) {
            const uint32_t k1 = (uint32_t)__builtin_ctz(word);
            word &= word - 1u;
            const bool two = word != 0u;
            const uint32_t k2 = two ? (uint32_t)__builtin_ctz(word) : k1;
            word &= word - 1u;  // (0 stays 0)
            const uint32_t j1 = base + k1, j2 = base + k2;
            const float4 a1 = rec[2 * (size_t)j1], b1 = rec[2 * (size_t)j1 + 1];
            const float4 a2 = rec[2 * (size_t)j2], b2 = rec[2 * (size_t)j2 + 1];
            const float3 q1 = make_float3(a1.x, a1.y, a1.z), q2 = make_float3(a2.x, a2.y, a2.z);
            const float3 v1 = make_float3(b1.x, b1.y, b1.z), v2 = make_float3(b2.x, b2.y, b2.z);
            const float2 d1 = make_float2(a1.w, b1.w), d2 = make_float2(a2.w, b2.w);
            // Keeps the second pair's loads beside the first pair's (one
            // memory round trip per iteration): without a use here the
            // compiler sinks them into the `two` branch below.
            asm volatile("" ::"v"(q2.x), "v"(q2.y), "v"(q2.z), "v"(v2.x), "v"(v2.y), "v"(v2.z), "v"(d2.x),
                         "v"(d2.y));
            pair_term_masked(A, pos, vel, pri, q1, v1, d1.x, d1.y, h, s);
            if (two) pair_term_masked(A, pos, vel, pri, q2, v2, d2.x, d2.y, h, s);
        }
        word = (uint32_t)(mm >> 32);  // then the high word
        base = first + 32u;
        if (!word) break;
    }
}

// One word of a row's mask over records staged in LDS (their first halves at
// st, their second halves at st + kStageRecs, so that 16-byte reads of
// consecutive records fall in distinct banks), bit k being record first + k,
// in ascending order, one per iteration: from LDS a pair's latency is covered
// by the SIMD's other wavefronts, and two pairs per iteration, the second
// one under a mask of its own, took 24% more cycles per row (6775 against
// 5466 SIMD cycles for a wavefront's nine rows of 24 neighbours).
__device__ __forceinline__ void walk_staged_word(PairAcc& A, uint32_t word, uint32_t first,
                                                 const float4* __restrict__ st, const float4& pos, const float4& vel,
                                                 float pri, float h, float s) {
    while (word) {
        const uint32_t j = first + (uint32_t)__builtin_ctz(word);
        word &= word - 1u;
        const float4 a = st[j], b = st[kStageRecs + j];
        pair_term_masked(A, pos, vel, pri, make_float3(a.x, a.y, a.z), make_float3(b.x, b.y, b.z), a.w, b.w, h, s);
    }
}

// The pairs of one row of forces_rowloop.
template <bool MASKS>
__device__ __forceinline__ void forces_row(PairAcc& A, uint32_t i, const float4& pos, const float4& vel, float pri,
                                           uint32_t rb, uint32_t re, unsigned long long mrow,
                                           const float4* __restrict__ rec, const float4* __restrict__ sp,
                                           const float4* __restrict__ sv, const float2* __restrict__ rho_p, float h,
                                           float s, float hhu) {
    if (MASKS && re - rb <= kRowMaskBits) {
        // the particle itself is in its own row's mask; it adds nothing
        if (i >= rb && i < re) mrow &= ~(1ull << (i - rb));
        walk_row_mask(A, mrow, rb, rec, pos, vel, pri, h, s);
    } else {
        for (uint32_t j = rb; j < re; j++)
            pair_term_rp(A, i, j, pos, vel, pri, ld_xyz(sp + j), ld_xyz(sv + j), rho_p[j], h, s, hhu);
    }
}

// The row loop of the force pass: the 9 stencil rows in turn, each row's
// neighbours from its mask (ascending, two per iteration) or, without a mask
// or for a row longer than 64 candidates, by re-testing every candidate.
template <bool MASKS>
__device__ __forceinline__ void forces_rowloop(PairAcc& A, uint32_t i, const float4& pos, const float4& vel,
                                               float2 dpi, const float4* __restrict__ sp,
                                               const float4* __restrict__ sv, const float2* __restrict__ rho_p,
                                               const uint32_t* __restrict__ start, const uint32_t* __restrict__ end,
                                               uint32_t n, const fg_common_fluid_params& cp, uint32_t key_base,
                                               const unsigned long long* __restrict__ masks) {
    const float h = cp.kernel_radius, hh = h * h;
    const float s = cp.simulation_scale;
    const float hu = h / s, hhu = hu * hu;
    const float cut = hh * 1.0001f;
    const RowWalker w = make_rows(pos, cp);
    const float4* rec = MASKS ? nbr_records(masks, n) : nullptr;
    for (int row = 0; row < 9; row++) {
        const int dz = row / 3 - 1, dy = row % 3 - 1;
        // The row's mask is read before its range is known, so the two
        // reads share one memory round trip (the asm keeps the compiler
        // from sinking the load behind the range test).
        unsigned long long mrow = 0ull;
        if (MASKS) {
            mrow = masks[(size_t)row * n + i];
            asm volatile("" ::"v"(mrow));
        }
        uint32_t rb, re;
        if (!row_range(w, dy, dz, cut, cp, key_base, start, end, n, rb, re)) continue;
        forces_row<MASKS>(A, i, pos, vel, dpi.y, rb, re, mrow, rec, sp, sv, rho_p, h, s, hhu);
    }
}

// The masked row loop for a whole wavefront (every lane present; a lane of an
// inactive particle, or one past the last particle, takes part with no rows)
// from the runs the density pass left: each row's neighbour records staged
// in the wavefront's LDS slice `stage` (kStageRecs first halves, then their
// second halves), the next row's records, masks and offsets loaded into
// registers while this row is walked.  Cells are looked up only for a row in
// which a lane has more candidates than its mask holds (it tests them where
// they are staged) and for one without a run.  Same pairs, same order, same
// sums as forces_rowloop<true>.
//
// Bound by VALU issue (3,342 instructions a wavefront) and by the records,
// which come from past the L2 cache three to four times at 8,388,608 particles
// (45% of a wavefront's time is waiting): 0.61 ms there against 0.76 with the
// cells looked up again and a min/max reduction per row; 80 against 94 us at
// 1,048,576.
//
// OTHER: with rows that lanes look up (kRunLong, kRunFar), a loop of its own,
// without loads ahead, so that the usual one keeps its registers (in one loop
// 1,048,576 particles took 178 us against 80).
template <bool OTHER>
__device__ __forceinline__ void forces_rows_staged(const WaveRuns& runs, PairAcc& A, uint32_t i, bool active, const float4& pos,
                                                   const float4& vel, float pri, const float4* __restrict__ sp,
                                                   const float4* __restrict__ sv, const float2* __restrict__ rho_p,
                                                   const uint32_t* __restrict__ start,
                                                   const uint32_t* __restrict__ end, uint32_t n,
                                                   const fg_common_fluid_params& cp, uint32_t key_base,
                                                   const unsigned long long* __restrict__ masks,
                                                   float4* __restrict__ stage) {
    const float h = cp.kernel_radius, s = cp.simulation_scale;
    const float hu = h / s, hhu = hu * hu;
    const uint32_t lane = __lane_id();
    const uint32_t wave = __builtin_amdgcn_readfirstlane(i >> 6);
    const float4* rec = nbr_records(masks, n);
    const uint16_t* offs = nbr_offs(masks, n) + (size_t)9 * 64 * wave + lane;
    float4 a0, b0, a1, b1;
    a0 = b0 = a1 = b1 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    unsigned long long next_mask = 0ull;
    uint32_t next_off = 0u;
    auto fetch = [&](int row) {
        const uint32_t len = runs.word(row) & kRunLength;
        next_mask = active ? masks[(size_t)row * n + i] : 0ull;
        next_off = offs[64 * row];
        const float4* q = rec + 2 * ((size_t)runs.first(row) + lane);
        if (lane < len) {
            a0 = q[0];
            b0 = q[1];
        }
        if (lane + 64u < len) {
            a1 = q[128];
            b1 = q[129];
        }
    };
    if (!OTHER) fetch(0);
    for (int row = 0; row < 9; row++) {
        const uint32_t word = runs.word(row), len = word & kRunLength, lo = runs.first(row);  // the same on every lane
        LaneRow r{0u, 0u};
        if (OTHER && (word & (kRunLong | kRunFar)))
            r = other_row(row, active, pos, lo, h * h * 1.0001f, cp, key_base, start, end, n);
        unsigned long long mm = OTHER ? (active ? masks[(size_t)row * n + i] : 0ull) : next_mask;
        const uint32_t off = OTHER ? offs[64 * row] : next_off;
        if (!OTHER && lane < len) {
            stage[lane] = a0;
            stage[kStageRecs + lane] = b0;
        }
        if (!OTHER && lane + 64u < len) {
            stage[lane + 64u] = a1;
            stage[kStageRecs + lane + 64u] = b1;
        }
        if (!OTHER && lane + 128u < min(len, kStageRecs)) {
            const float4* q = rec + 2 * ((size_t)lo + lane + 128u);
            stage[lane + 128u] = q[0];
            stage[kStageRecs + lane + 128u] = q[1];
        }
        for (uint32_t k = lane; OTHER && k < min(len, kStageRecs); k += 64u) {
            const float4* q = rec + 2 * ((size_t)lo + k);
            stage[k] = q[0];
            stage[kStageRecs + k] = q[1];
        }
        if (!OTHER && row < 8) fetch(row + 1);
        LaneRow test{0u, 0u};  // the lane's candidates where its mask does not hold them
        if (OTHER && (word & (kRunLong | kRunFar))) {
            if (word & kRunFar) {  // from memory, one by one: two at a time need more registers than the loop has
                const uint32_t rb = lo + r.off;
                if (r.len > kRowMaskBits) mm = 0ull;
                for (uint32_t k = 0u; k < r.len; k++) {
                    if (r.len <= kRowMaskBits) {
                        if (mm == 0ull) break;
                        k = (uint32_t)__builtin_ctzll(mm);
                        mm &= mm - 1ull;
                    }
                    const float4 a = rec[2 * (size_t)(rb + k)], b = rec[2 * (size_t)(rb + k) + 1];
                    pair_term(A, i, rb + k, pos, vel, pri, make_float3(a.x, a.y, a.z), make_float3(b.x, b.y, b.z), a.w,
                              b.w, h, s, hhu);
                }
                continue;
            }
            if (r.len > kRowMaskBits) {
                test = r;
                mm = 0ull;
            }
        }
        // the particle itself is in its own cell's row; it adds nothing
        if (row == 4) mm &= ~(1ull << ((i - lo - off) & 63u));
        wave_lds_sync();
        if (len <= kStageRecs && !(OTHER && (word & kRunLong))) {
            walk_staged_word(A, (uint32_t)mm, off, stage, pos, vel, pri, h, s);
            if (word & kRunWide) walk_staged_word(A, (uint32_t)(mm >> 32), off + 32u, stage, pos, vel, pri, h, s);
            wave_lds_sync();  // every lane's reads before the next stores
            continue;
        }
        // A run that fills the slice more than once: the mask is walked as far
        // as the records [at, at + kStageRecs) of the run go, then on from there,
        // and so are the candidates to test.
        for (uint32_t at = 0u;;) {
            while (mm) {
                const uint32_t j = off + (uint32_t)__builtin_ctzll(mm) - at;
                if (j >= kStageRecs) break;
                mm &= mm - 1ull;
                const float4 a = stage[j], b = stage[kStageRecs + j];
                pair_term_masked(A, pos, vel, pri, make_float3(a.x, a.y, a.z), make_float3(b.x, b.y, b.z), a.w, b.w, h,
                                 s);
            }
            const uint32_t last = min(test.off + test.len, at + kStageRecs);
            for (uint32_t k = max(test.off, at); OTHER && k < last; k++) {
                const float4 a = stage[k - at], b = stage[kStageRecs + k - at];
                pair_term(A, i, lo + k, pos, vel, pri, make_float3(a.x, a.y, a.z), make_float3(b.x, b.y, b.z), a.w, b.w,
                          h, s, hhu);
            }
            wave_lds_sync();
            at += kStageRecs;
            if (at >= len) break;
            for (uint32_t k = lane; k < min(len - at, kStageRecs); k += 64u) {
                const float4* q = rec + 2 * ((size_t)lo + at + k);
                stage[k] = q[0];
                stage[kStageRecs + k] = q[1];
            }
            wave_lds_sync();
        }
    }
}

// A wavefront's slice in the force pass without masks: the records of the
// current part of a run, (x, y), (z, 1/rho) and (vx, vy, vz, p/rho) apart, so
// that the distance test reads them as the density pass does.
struct ForceStage {
    float2 xy[kStageRecs + 4], za[kStageRecs + 4];
    float4 vb[kStageRecs];
    WaveCells cells;
    __device__ __forceinline__ uint32_t* temp() { return reinterpret_cast<uint32_t*>(xy); }
};
static_assert(offsetof(ForceStage, cells) >= sizeof(uint32_t) * kWaveCellsTemp, "wave_cells' temporary words");

// The bits of up to 32 staged candidates from slice index `at` that lie
// within h of p (density_group's hit bits; p and the slice hold no NaN).
#pragma clang fp contract(off)
__device__ __forceinline__ uint32_t near_bits(const float4& p, const ForceStage& st, uint32_t at, uint32_t cnt,
                                              float hhu) {
    const float2* xy = st.xy + at;
    const float2* za = st.za + at;
    uint32_t bits = 0u, k = 0u;
    for (; k < cnt; k += 4u) {
#pragma unroll
        for (uint32_t u = 0; u < 4u; u++) {
            const float dx = p.x - xy[k + u].x, dy = p.y - xy[k + u].y, dz = p.z - za[k + u].x;
            const float r2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
            bits = __builtin_amdgcn_alignbit(bits, __float_as_uint(r2 - hhu), 31);
        }
    }
    const uint32_t word = __builtin_bitreverse32(bits) >> (32u - k);
    return cnt < 32u ? word & ((1u << cnt) - 1u) : word;  // (what lies past them in the slice)
}
#pragma clang fp contract(fast)

// The row loop without masks for a whole wavefront (as forces_rows_staged):
// each row's records are made from the sorted arrays while they are staged,
// the lanes test their candidates there and then walk those within h.  Same
// pairs, same order, same sums as forces_rowloop<false>.
//
// Bound by VALU issue (the test and the walk); 250,047 particles take 48 us,
// where every candidate's position, velocity and density read from memory
// and a division per candidate took 97; 1,048,576 take 159, then 344.
template <bool OTHER>
__device__ __forceinline__ void forces_rows_tested(const WaveRuns& runs, const RowWalker& w, uint32_t cell, PairAcc& A,
                                                   uint32_t i, bool active, const float4& pos,
                                                   const float4& vel, float pri, const float4* __restrict__ sp,
                                                   const float4* __restrict__ sv, const float2* __restrict__ rho_p,
                                                   const uint32_t* __restrict__ start,
                                                   const uint32_t* __restrict__ end, uint32_t n,
                                                   const fg_common_fluid_params& cp, uint32_t key_base,
                                                   ForceStage& st) {
    const float h = cp.kernel_radius, s = cp.simulation_scale;
    const float hu = h / s, hhu = hu * hu, cut = h * h * 1.0001f;
    const uint32_t lane = __lane_id();
    const bool walks = active && finite_position(pos);
    float3 p0, p1, v0, v1;
    float2 d0, d1;
    p0 = p1 = v0 = v1 = make_float3(0.0f, 0.0f, 0.0f);
    d0 = d1 = make_float2(1.0f, 0.0f);
    auto load = [&](uint32_t j, float3& p, float3& v, float2& d) {
        p = ld_xyz(sp + j);
        v = ld_xyz(sv + j);
        d = rho_p[j];
    };
    auto put = [&](uint32_t k, const float3& p, const float3& v, const float2& d) {
        const float a = 1.0f / d.x;
        st.xy[k] = make_float2(stage_number(p.x), stage_number(p.y));
        st.za[k] = make_float2(stage_number(p.z), a);
        st.vb[k] = make_float4(v.x, v.y, v.z, d.y * a);
    };
    auto fetch = [&](int row) {
        const uint32_t len = runs.word(row) & kRunLength, lo = runs.first(row);
        if (lane < len) load(lo + lane, p0, v0, d0);
        if (lane + 64u < len) load(lo + lane + 64u, p1, v1, d1);
    };
    fetch(0);
    for (int row = 0; row < 9; row++) {
        const uint32_t info = runs.word(row), len = info & kRunLength, lo = runs.first(row);  // the same on every lane
        LaneRow r = lane_row(st.cells, row, cell, walks, w, cut);
        if (OTHER && (info & (kRunLookup | kRunFar)))
            r = other_row(row, walks, pos, lo, cut, cp, key_base, start, end, n);
        if (OTHER && (info & kRunFar)) {
            if (r.len)
                forces_row<false>(A, i, pos, vel, pri, lo + r.off, lo + r.off + r.len, 0ull, nullptr, sp, sv, rho_p, h, s,
                                  hhu);
            r.len = 0u;
        }
        for (uint32_t at = 0u;;) {  // (a run rarely fills the slice)
            const uint32_t cnt = min(len - at, kStageRecs);
            if (at == 0u) {
                if (lane < cnt) put(lane, p0, v0, d0);
                if (lane + 64u < cnt) put(lane + 64u, p1, v1, d1);
                if (row < 8) fetch(row + 1);
            }
            for (uint32_t k = lane + (at == 0u ? 128u : 0u); k < cnt; k += 64u) {
                float3 p, v;
                float2 d;
                load(lo + at + k, p, v, d);
                put(k, p, v, d);
            }
            wave_lds_sync();
            const uint32_t b = min(r.off + r.len, at + kStageRecs);
            for (uint32_t a = max(r.off, at); a < b; a += 32u) {
                const uint32_t c = min(b - a, 32u), k0 = a - at;
                uint32_t word = near_bits(pos, st, k0, c, hhu);
                const uint32_t self = i - (lo + a);  // the particle itself adds nothing
                if (self < 32u) word &= ~(1u << self);
                while (word) {
                    const uint32_t k = k0 + (uint32_t)__builtin_ctz(word);
                    word &= word - 1u;
                    const float2 xy = st.xy[k], za = st.za[k];
                    const float4 vb = st.vb[k];
                    pair_term_masked(A, pos, vel, pri, make_float3(xy.x, xy.y, za.x), make_float3(vb.x, vb.y, vb.z),
                                     za.y, vb.w, h, s);
                }
            }
            wave_lds_sync();  // every lane's reads before the next stores
            at += kStageRecs;
            if (at >= len) break;
        }
    }
}

// `v`; with LATER, by a pointer that the compiler takes for a new one, so that
// nothing read through it is read before this point.
template <bool LATER, class T>
__device__ __forceinline__ const T& later(const T& v) {
    if constexpr (LATER) {
        const T* p = &v;
        asm volatile("" : "+s"(p));
        return *p;
    } else {
        return v;
    }
}

// Per-lane row table of the flat force schedule, in LDS: for each of the 9
// stencil rows, the sorted index of its first particle and its neighbour
// mask (0 for a culled row).  The flat schedule takes rows of at most 32
// candidates, so a mask is one 32-bit word: 72 bytes per lane, which keeps
// eight 256-lane workgroups' tables within a CU's LDS.
constexpr uint32_t kFlatRowBits = 32;
struct FlatRows {
    uint32_t* rb;  // [9][lanes]
    uint32_t* mm;  // [9][lanes]
    uint32_t lanes, lane;
    __device__ __forceinline__ uint32_t& b(int r) { return rb[r * lanes + lane]; }
    __device__ __forceinline__ uint32_t& m(int r) { return mm[r * lanes + lane]; }
};

// Pressure + viscosity + walls (+ body contact) of sorted particle i (i < n),
// written to vout[id[i]] (and pout[id[i]] when integrating).
//
// Two schedules give bit-identical sums (rows in order, neighbours of a row
// in ascending sorted order):
//  * row loop: the 9 rows in turn; a wavefront waits at every row for its
//    lane with the most neighbours in that row.  Given an LDS slice
//    (`stage`) and a whole wavefront, each row's records are staged there
//    first (forces_rows_staged); its last lanes may have i >= n and then
//    only take part;
//  * flat (MASKS with a row table): the rows with neighbours are gathered
//    first, compacted in row order, then each lane walks its own neighbour
//    stream across them, two neighbours per iteration with their loads
//    issued together, so a wavefront runs for its lane with the most
//    neighbours overall rather than, row by row, for the lane with the
//    most neighbours in that row.  The next row's entry is read from LDS
//    one row ahead.  A particle with a row longer than kFlatRowBits takes
//    the row loop.
//
// INDIRECT: cp lies in memory at a wave-uniform address (a batch's scene):
// what follows the pair sums then reads it through a pointer of its own, or
// the compiler loads all of it up front and keeps it in vector registers
// during the pair sums.
template <bool MASKS, bool COUPLED = false, bool DEFER = false, bool INDIRECT = false>
__device__ __forceinline__ void forces_particle(uint32_t i, const float4* __restrict__ sp,
                                                const float4* __restrict__ sv, const float2* __restrict__ rho_p,
                                                const uint32_t* __restrict__ start, const uint32_t* __restrict__ end,
                                                float4* __restrict__ vout, float4* __restrict__ pout,
                                                const uint32_t* __restrict__ id, uint32_t n, float m, float mu,
                                                const fg_common_fluid_params& cp0, const fg_kernels_cache& kc0,
                                                uint32_t key_base, const unsigned long long* __restrict__ masks,
                                                const Contacts& bc, FlatRows* flat = nullptr,
                                                const DeferredContact* defer = nullptr,
                                                float4* __restrict__ stage = nullptr, ForceStage* tested = nullptr) {
    const uint32_t il = flat ? i : min(i, n - 1u);
    const float4 pos = sp[il];
    const float4 vel = sv[il];
    const bool active = i < n && pos.w > 0.0f;
    F3 a = f3(0.0f, 0.0f, 0.0f);
    PairAcc A{0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    // The staged row loop needs every lane of the wavefront, as the density
    // pass did; otherwise the rows are read from memory below.
    bool staged_rows = false;
    if (MASKS && stage != nullptr && flat == nullptr && __ballot(1) == ~0ull) {
        const float pri = rho_p[il].y;
        const uint32_t lane = __lane_id();
        WaveRuns runs;
        if (lane < 9u) {
            const uint32_t* t = nbr_runs(masks, n) + (size_t)kRunWords * __builtin_amdgcn_readfirstlane(i >> 6) + lane;
            runs.lo = t[0];
            runs.info = t[9];
        }
        if (__ballot((runs.info & (kRunLong | kRunFar)) != 0u) == 0ull)
            forces_rows_staged<false>(runs, A, i, active, pos, vel, pri, sp, sv, rho_p, start, end, n, cp0, key_base,
                                      masks, stage);
        else
            forces_rows_staged<true>(runs, A, i, active, pos, vel, pri, sp, sv, rho_p, start, end, n, cp0, key_base,
                                     masks, stage);
        staged_rows = true;
    }
    if (!MASKS && tested != nullptr && __ballot(1) == ~0ull) {
        const float pri = rho_p[il].y;
        const RowWalker w = make_rows(pos, cp0);
        uint32_t cell;
        WaveRuns runs;
        wave_cells(tested->cells, tested->temp(), 64u, w, cp0, key_base, start, end, n, cell, runs);
        if (__builtin_expect(__ballot((runs.info & (kRunLookup | kRunFar)) != 0u) == 0ull, 1))
            forces_rows_tested<false>(runs, w, cell, A, i, active, pos, vel, pri, sp, sv, rho_p, start, end, n, cp0, key_base,
                                      *tested);
        else
            forces_rows_tested<true>(runs, w, cell, A, i, active, pos, vel, pri, sp, sv, rho_p, start, end, n, cp0, key_base,
                                     *tested);
        staged_rows = true;
    }
    const fg_common_fluid_params& cp = later<INDIRECT>(cp0);
    const fg_kernels_cache& kc = later<INDIRECT>(kc0);
    if (i >= n) return;
    if (active) {
        const float h = cp.kernel_radius, hh = h * h;
        const float s = cp.simulation_scale;
        const float cut = hh * 1.0001f;
        const float2 dpi = rho_p[i];
        const RowWalker w = make_rows(pos, cp);
        const float4* rec = MASKS ? nbr_records(masks, n) : nullptr;
        bool rowloop = !staged_rows;
        if (MASKS && flat) {
            // The rows with neighbours, compacted in row order: (first sorted
            // index, mask without the particle itself).
            bool fits = true;
            uint32_t nrows = 0;
#pragma unroll
            for (int row = 0; row < 9; row++) {
                const int dz = row / 3 - 1, dy = row % 3 - 1;
                uint32_t rb = 0, re = 0;
                if (row_range(w, dy, dz, cut, cp, key_base, start, end, n, rb, re)) {
                    if (re - rb <= kFlatRowBits) {
                        unsigned long long m64 = masks[(size_t)row * n + i];
                        // the particle itself is in its own row's mask; it adds nothing
                        if (i >= rb && i < re) m64 &= ~(1ull << (i - rb));
                        const uint32_t mm = (uint32_t)m64;
                        if (mm) {
                            flat->b(nrows) = rb;
                            flat->m(nrows) = mm;
                            nrows++;
                        }
                    } else {
                        fits = false;
                    }
                }
            }
            if (fits) {
                rowloop = false;
                // cm/cb: the current row's remaining mask and first index;
                // nm/nb: the next row's, read from LDS one row ahead.
                uint32_t k = 0;
                uint32_t cm = nrows > 0 ? flat->m(0) : 0u, cb = nrows > 0 ? flat->b(0) : 0u;
                uint32_t nm = nrows > 1 ? flat->m(1) : 0u, nb = nrows > 1 ? flat->b(1) : 0u;
                // The next neighbour of the stream (cm != 0 on entry).
                auto next = [&]() -> uint32_t {
                    const uint32_t j = cb + (uint32_t)__builtin_ctz(cm);
                    cm &= cm - 1u;
                    if (cm == 0u) {
                        cm = nm;
                        cb = nb;
                        k++;
                        nm = k + 1 < nrows ? flat->m(k + 1) : 0u;
                        nb = k + 1 < nrows ? flat->b(k + 1) : 0u;
                    }
                    return j;
                };
                while (cm != 0u) {
                    const uint32_t j1 = next();
                    const bool two = cm != 0u;
                    const uint32_t j2 = two ? next() : j1;
                    const float4 a1 = rec[2 * (size_t)j1], b1 = rec[2 * (size_t)j1 + 1];
                    const float4 a2 = rec[2 * (size_t)j2], b2 = rec[2 * (size_t)j2 + 1];
                    const float3 q1 = make_float3(a1.x, a1.y, a1.z), q2 = make_float3(a2.x, a2.y, a2.z);
                    const float3 v1 = make_float3(b1.x, b1.y, b1.z), v2 = make_float3(b2.x, b2.y, b2.z);
                    const float2 d1 = make_float2(a1.w, b1.w), d2 = make_float2(a2.w, b2.w);
                    asm volatile("" ::"v"(q2.x), "v"(q2.y), "v"(q2.z), "v"(v2.x), "v"(v2.y), "v"(v2.z), "v"(d2.x),
                                 "v"(d2.y));
                    pair_term_masked(A, pos, vel, dpi.y, q1, v1, d1.x, d1.y, h, s);
                    if (two) pair_term_masked(A, pos, vel, dpi.y, q2, v2, d2.x, d2.y, h, s);
                }
            }
        }
        if (rowloop) forces_rowloop<MASKS>(A, i, pos, vel, dpi, sp, sv, rho_p, start, end, n, cp, key_base, masks);
        // pressure: (s d_u / r) = d_u / r_u, so no scale factor remains
        const float iri = 1.0f / dpi.x;
        const float cP = -kc.kSpikyGradient * iri;
        const float cV = kc.kViscosityLaplacian * mu * iri;
        const F3 internal = f3(__builtin_fmaf(cP, A.px, cV * A.vx), __builtin_fmaf(cP, A.py, cV * A.vy),
                               __builtin_fmaf(cP, A.pz, cV * A.vz));
        if (DEFER && bc.coupled && contact_possible(pos, bc)) {
            defer_particle(*defer, i, internal);
            return;
        }
        a = DEFER ? finish_accel<true, true>(internal, m, pos, vel, cp, bc)
                  : finish_accel<COUPLED>(internal, m, pos, vel, cp, bc);
    }
    write_back(id[i], n, pos, vel, a, cp, vout, pout);
}

}  // namespace fg
