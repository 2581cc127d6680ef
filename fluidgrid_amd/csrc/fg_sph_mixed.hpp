// fg_sph_mixed.hpp -- the mixed-precision density pass (LINEAR keys, fast
// math): candidates are culled two at a time in packed FP16 from 8-byte
// cell-relative offsets, and the survivors are evaluated exactly as the FP32
// pass evaluates every candidate, with a compensated (Neumaier) sum.
//
// Offsets.  For a particle in LINEAR cell (cx, cy, cz), with lower corner lo
// and u_a = clamp((x_a - lo_a) / cs_a, 0, 1) its position inside the cell
// (clamped: a particle outside the grid is projected onto its clamped cell),
// in units of the largest cell edge L (w_a = cs_a / L):
//     X = w_x (u_x + (cx mod 3) - 1.5),  Y = w_y (u_y - 0.5),  Z = w_z (u_z - 0.5).
// A stencil row holds the cells cx-1..cx+1 at (cy+dy, cz+dz).  For a
// candidate j of that row, Y_j - (Y_i - dy w_y) is the y distance of the two
// projections, likewise z.  X_j - X_i is their x distance up to a multiple
// of the period P = 3 w_x (the cells' indices are only known mod 3); the
// distance is min(|X_j - X_i|, P - |X_j - X_i|), exact whenever the true x
// distance is at most P/2 = 1.5 w_x, which every pair within h satisfies
// (h <= cs_x, the stencil's own requirement).
//
// Conservative cull.  Projection onto a box is 1-Lipschitz, so the projected
// distance never exceeds the true one.  The FP16 evaluation adds at most, in
// L^2 units, 8.4e-3 to r^2 for pairs with r <= h:
//   stored X, Y, Z: |.| <= 1.5, rounding <= 2^-11; the row shifts
//   (|.| <= 1.5): <= 2^-11; the differences (|.| < 3): <= 2^-10; P: <= 2^-10
//   (P - a is exact where it is taken, a in [P/2, P]); so each component is
//   off by at most e = 2^-9;
//   r^2 = fma(dz, dz, fma(dy, dy, fma(dx, dx, -cut))): with |d| <= 1 the
//   components add at most 2 e (|dx| + |dy| + |dz|) <= 2 sqrt(3) e = 6.8e-3,
//   and the three roundings (results below 2) 3 * 2^-11 = 1.5e-3;
// plus the FP32 cell and offset arithmetic (below 1e-4).  The cut is
// (h/L)^2 + 2^-6 (1.6e-2), rounded up, so no pair that the FP32 test accepts
// is culled: the survivors' exact test then sets exactly the row-mask bits
// of the FP32 pass, and the force pass reads the same masks.
#pragma once
#include "fg_sph_tile.hpp"

namespace fg {

typedef _Float16 half2v __attribute__((ext_vector_type(2)));

struct HalfGeom {
    float ix, iy, iz;  // 1 / cell size
    float wx, wy, wz;  // cell size / L
    float per;         // 3 w_x
    float cut;         // (h/L)^2 + 2^-6, rounded up past FP16 rounding
};

__device__ __forceinline__ HalfGeom half_geom(const fg_common_fluid_params& cp) {
    HalfGeom g;
    const float L = fmaxf(cp.cell_size.x, fmaxf(cp.cell_size.y, cp.cell_size.z));
    g.ix = 1.0f / cp.cell_size.x;
    g.iy = 1.0f / cp.cell_size.y;
    g.iz = 1.0f / cp.cell_size.z;
    g.wx = cp.cell_size.x / L;
    g.wy = cp.cell_size.y / L;
    g.wz = cp.cell_size.z / L;
    g.per = 3.0f * g.wx;
    const float hc = (cp.kernel_radius / cp.simulation_scale) / L;
    g.cut = (hc * hc + 0.015625f) * 1.001953125f;  // x (1 + 2^-9) covers the FP16 rounding of the cut
    return g;
}

// The offsets (X, Y, Z) of a particle at p, in FP32.
__device__ __forceinline__ float3 half_offsets(const float4& p, const fg_common_fluid_params& cp,
                                               const HalfGeom& g) {
    const CellXYZ c = linear_cell(p.x, p.y, p.z, cp);
    const float lx = cp.volume_min.x + (float)c.x * cp.cell_size.x;
    const float ly = cp.volume_min.y + (float)c.y * cp.cell_size.y;
    const float lz = cp.volume_min.z + (float)c.z * cp.cell_size.z;
    // fmaxf first: a NaN coordinate becomes 0 (its exact tests fail anyway)
    const float ux = fminf(fmaxf((p.x - lx) * g.ix, 0.0f), 1.0f);
    const float uy = fminf(fmaxf((p.y - ly) * g.iy, 0.0f), 1.0f);
    const float uz = fminf(fmaxf((p.z - lz) * g.iz, 0.0f), 1.0f);
    return make_float3(g.wx * (ux + (float)(c.x % 3) - 1.5f), g.wy * (uy - 0.5f), g.wz * (uz - 0.5f));
}

__device__ __forceinline__ uint32_t pack_half2(float lo, float hi) {
    const half2v v = {(_Float16)lo, (_Float16)hi};
    return __builtin_bit_cast(uint32_t, v);
}

// Pair record r of the sorted particles: (X_r, X_r+1), (Y_r, Y_r+1),
// (Z_r, Z_r+1), 0 as packed FP16; records n and n+1 are zero (reads past a
// row's end are masked off).
__device__ __forceinline__ uint4* nbr_half(unsigned long long* masks, uint32_t n) {
    return reinterpret_cast<uint4*>(reinterpret_cast<char*>(masks) + nbr_half_offset(n));
}
__device__ __forceinline__ const uint4* nbr_half(const unsigned long long* masks, uint32_t n) {
    return reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(masks) + nbr_half_offset(n));
}

#pragma clang fp contract(off)
// r^2 - cut of the two candidates of a pair record, packed; a candidate
// survives when its half is negative.
__device__ __forceinline__ uint32_t cull_pair(const uint4& r, half2v tx, half2v ty, half2v tz, half2v per,
                                              half2v ncut) {
    const half2v X = __builtin_bit_cast(half2v, r.x);
    const half2v Y = __builtin_bit_cast(half2v, r.y);
    const half2v Z = __builtin_bit_cast(half2v, r.z);
    const half2v a = __builtin_elementwise_abs(X - tx);
    const half2v dx = __builtin_elementwise_min(a, per - a);
    const half2v dy = Y - ty, dz = Z - tz;
    const half2v d = __builtin_elementwise_fma(dz, dz, __builtin_elementwise_fma(dy, dy,
                                               __builtin_elementwise_fma(dx, dx, ncut)));
    return __builtin_bit_cast(uint32_t, d);
}

// Shifts the survivor bits of a pair record's two candidates into `bits` from
// below, the first candidate first: the halves' signs.
__device__ __forceinline__ uint32_t push_pair(uint32_t bits, uint32_t d) {
    bits = __builtin_amdgcn_alignbit(bits, d << 16, 31);
    return __builtin_amdgcn_alignbit(bits, d, 31);
}

// |p - q|^2 with the operations of density4 (the FP32 pass's test).
__device__ __forceinline__ float exact_r2(const float4& p, const float3& q) {
    const float dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
    return __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
}
__device__ __forceinline__ float poly6_term(float h2u, float r2) {
    const float t = h2u - r2;
    return (t * t) * t;
}

// sum + comp += x (Neumaier's compensated summation), for a sum and an x that
// are not negative: which is larger in magnitude is then one plain compare.  (A
// term that the rounding of h^2 leaves just below zero is exact in both forms.)
__device__ __forceinline__ void neumaier_add(float& sum, float& comp, float x) {
    const float t = sum + x;
    comp += (sum >= x) ? ((sum - t) + x) : ((x - t) + sum);
    sum = t;
}
#pragma clang fp contract(fast)

// A wavefront's staged run: the pair records (the two after the run too: a
// group of candidates t..t+3 reads the records t and t + 2) and the positions,
// each as 8 and 4 bytes: lanes read at unrelated offsets, and 16-byte reads of
// that kind take three to four times the LDS cycles of an 8- and a 4-byte one.
//
// Bound by VALU issue: 5,770 instructions a wavefront against the FP32 pass's
// 4,670, and more of them (packed FP16, compares, selects, bit moves) of those
// that take 4 cycles and more to issue, so a packed pair of candidates costs
// what two FP32 ones do.  2,097,152 particles: the step 595 us with 16-byte
// staging in workgroups of 256, rows loaded when they are needed and survivors
// four at a time, 585 us so.
constexpr uint32_t kMixedStage = 128;
struct MixedStage {
    uint2 hxy[kMixedStage + 2];
    float2 xy[kMixedStage];
    uint32_t hz[kMixedStage + 2];
    float z[kMixedStage];
    WaveCells cells;
};
static_assert(offsetof(MixedStage, cells) >= sizeof(uint32_t) * kWaveCellsTemp, "wave_cells' temporary words");

// One stencil row of the mixed density pass for one particle: the cull of
// the row's candidates from their FP16 pair records, then the exact FP32
// test and compensated sum of the survivors.  `at` is the row's first
// candidate, in the staged run or (LDS false) among the sorted arrays.
struct MixedRow {
    float4 p;
    half2v tx, per, ncut;
    float hhu, h2u;
    float sum, comp;
    const MixedStage& st;
    const uint4* __restrict__ H;
    const float4* __restrict__ P;

    // The survivors among the candidates at + (bits of word); returns the bits
    // of those within h (the FP32 test of density4).  One an iteration from LDS,
    // two from memory, whose loads are then in flight together (1,048,576
    // particles on cells of 2 h 538 us, one by one 566, by four 592).
    template <bool LDS>
    __device__ __forceinline__ uint32_t exact(uint32_t word, uint32_t at) {
        constexpr int N = LDS ? 1 : 2;
        uint32_t hits = 0u;
        while (word) {
            uint32_t bit[N];
            float3 q[N];
#pragma unroll
            for (int u = 0; u < N; u++) {
                const uint32_t rest = word & (word - 1u), k = u == 0 || word ? (uint32_t)__builtin_ctz(word) : 0u;
                bit[u] = word ^ rest;
                word = rest;
                if (LDS) {
                    const float2 xy = st.xy[at + k];
                    q[u] = make_float3(xy.x, xy.y, st.z[at + k]);
                } else
                    q[u] = ld_xyz(P + at + k);
            }
#pragma unroll
            for (int u = 0; u < N; u++) {
                const float r2 = exact_r2(p, q[u]);
                const bool hit = r2 < hhu && (u == 0 || bit[u] != 0u);
                neumaier_add(sum, comp, hit ? poly6_term(h2u, r2) : 0.0f);
                hits |= hit ? bit[u] : 0u;
            }
        }
        return hits;
    }

    // Survivor bits of the cnt (<= 32) candidates from `at`.
    template <bool LDS>
    __device__ __forceinline__ uint32_t cull_word(uint32_t at, uint32_t cnt, half2v ty, half2v tz) const {
        uint32_t bits = 0u, t = 0u;
        for (; t < cnt; t += 4) {
            uint4 r0, r1;
            if (LDS) {
                const uint2 a = st.hxy[at + t], b = st.hxy[at + t + 2];
                r0 = make_uint4(a.x, a.y, st.hz[at + t], 0u);
                r1 = make_uint4(b.x, b.y, st.hz[at + t + 2], 0u);
            } else {
                r0 = H[at + t];
                r1 = H[at + t + 2];
            }
            bits = push_pair(bits, cull_pair(r0, tx, ty, tz, per, ncut));
            bits = push_pair(bits, cull_pair(r1, tx, ty, tz, per, ncut));
        }
        if (t == 0u) return 0u;
        const uint32_t word = __builtin_bitreverse32(bits) >> (32u - t);  // candidate j was shifted in as bit t - 1 - j
        return cnt < 32u ? word & ((1u << cnt) - 1u) : word;
    }

    // The row's mask: 64 candidates at a time; a row longer than 64 is never
    // read through its mask (the force pass re-tests it), which is 0.
    template <bool LDS>
    __device__ __forceinline__ unsigned long long row(uint32_t at, uint32_t len, half2v ty, half2v tz) {
        unsigned long long msk = 0ull;
        for (uint32_t c0 = 0; c0 < len; c0 += 32u) {
            const uint32_t w = cull_word<LDS>(at + c0, min(len - c0, 32u), ty, tz);
            msk |= (unsigned long long)exact<LDS>(w, at + c0) << (c0 & 32u);
        }
        return len > kRowMaskBits ? 0ull : msk;
    }
};

// Density of sorted particle i (i < n) in the mixed form: the row masks and
// the neighbour record of the FP32 pass (density_particle<true>), and
// rho = m kPoly6 s^6 sum (h^2 - r^2)^3 over the same pairs, summed in
// ascending sorted order within rows in order, compensated.
//
// Given an LDS slice (`stage`) and a whole wavefront, each row's run of pair
// records and positions is staged there first, as in density_rows_staged;
// every lane then takes part (the lane of an inactive particle, or one past
// the last particle, with no rows), and the runs are left for the force pass.
__device__ __forceinline__ void density_particle_mixed(uint32_t i, const float4* __restrict__ sp,
                                                       const float4* __restrict__ sv, float2* __restrict__ rho_p,
                                                       const uint32_t* __restrict__ start,
                                                       const uint32_t* __restrict__ end, uint32_t n, float k,
                                                       float rho0, float m, const fg_common_fluid_params& cp,
                                                       const fg_kernels_cache& kc,
                                                       unsigned long long* __restrict__ masks, MixedStage& st) {
    const bool valid = i < n;
    const uint32_t il = min(i, n - 1u), lane = __lane_id();
    const float4 p = sp[il];
    float4* rec = nbr_records(masks, n);
    const bool active = valid && p.w > 0.0f;
    const float s = cp.simulation_scale, s2 = s * s;
    const float h = cp.kernel_radius, hh = h * h;
    const float hu = h / s, hhu = hu * hu, h2u = cp.kernel_radius_squared / s2;
    const float cut = hh * 1.0001f;
    const RowWalker w = make_rows(p, cp);
    uint32_t cell, words = 0u;
    WaveRuns runs;
    wave_cells(st.cells, reinterpret_cast<uint32_t*>(st.hxy), 64u, w, cp, 0u, start, end, n, cell, runs);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(i >> 6);
    const bool table = n >= kRunMinParticles;
    uint16_t* offs = nbr_offs(masks, n) + (size_t)9 * 64 * wave + lane;
    const HalfGeom g = half_geom(cp);
    const float3 o = half_offsets(p, cp, g);
    const uint4* __restrict__ hr = nbr_half(masks, n);
    MixedRow M{p,
               half2v{(_Float16)o.x, (_Float16)o.x},
               half2v{(_Float16)g.per, (_Float16)g.per},
               half2v{(_Float16)(-g.cut), (_Float16)(-g.cut)},
               hhu,
               h2u,
               0.0f,
               0.0f,
               st,
               hr,
               sp};
    // the next row's records and positions, loaded while a row is walked
    uint4 h0 = make_uint4(0u, 0u, 0u, 0u), h1 = h0;
    float3 p0 = make_float3(0.0f, 0.0f, 0.0f), p1 = p0;
    auto fetch = [&](int row) {
        const uint32_t len = runs.word(row) & kRunLength, lo = runs.first(row);
        if (len > kMixedStage) return;
        if (lane < len + 2u) h0 = hr[lo + lane];
        if (lane + 64u < len + 2u) h1 = hr[lo + lane + 64u];
        if (lane < len) p0 = ld_xyz(sp + lo + lane);
        if (lane + 64u < len) p1 = ld_xyz(sp + lo + lane + 64u);
    };
    auto put = [&](uint32_t q, const uint4& h, const float3& pos, bool candidate) {
        st.hxy[q] = make_uint2(h.x, h.y);
        st.hz[q] = h.z;
        if (candidate) {
            st.xy[q] = make_float2(pos.x, pos.y);
            st.z[q] = pos.z;
        }
    };
    fetch(0);

    for (int row = 0; row < 9; row++) {
        const int dz = row / 3 - 1, dy = row % 3 - 1;
        const uint32_t info = runs.word(row), len = info & kRunLength, lo = runs.first(row);  // the same on every lane
        const bool staged = len <= kMixedStage && !(info & kRunFar);
        LaneRow r = lane_row(st.cells, row, cell, active, w, cut);
        if (info & (kRunLookup | kRunFar)) r = other_row(row, active, p, lo, cut, cp, 0u, start, end, n);
        const bool has = r.len != 0u;
        const uint32_t rb = lo + r.off, re = rb + r.len;
        if (table) {
            offs[64 * row] = (uint16_t)r.off;
            const uint32_t word = run_word(info, r.len);
            words = (int)lane == row ? word : words;
        }
        if (staged) {
            if (lane < len + 2u) put(lane, h0, p0, lane < len);
            if (lane + 64u < len + 2u) put(lane + 64u, h1, p1, lane + 64u < len);
            if (lane + 128u < len + 2u) put(lane + 128u, hr[lo + lane + 128u], p0, false);
            wave_lds_sync();
        }
        if (row < 8) fetch(row + 1);
        unsigned long long msk = 0ull;
        if (has) {
            const half2v ty = {(_Float16)(o.y - (float)dy * g.wy), (_Float16)(o.y - (float)dy * g.wy)};
            const half2v tz = {(_Float16)(o.z - (float)dz * g.wz), (_Float16)(o.z - (float)dz * g.wz)};
            msk = staged ? M.row<true>(rb - lo, re - rb, ty, tz) : M.row<false>(rb, re - rb, ty, tz);
        }
        if (active) masks[(size_t)row * n + i] = msk;
        if (staged) wave_lds_sync();  // every lane's reads of this row before the next row's stores
    }
    if (table) {
        runs.info = words;
        store_runs(runs, wave, masks, n);
    }
    if (!valid) return;
    const float4 v = sv[i];
    if (active)
        store_density(i, m * kc.kPoly6 * (s2 * s2 * s2) * (M.sum + M.comp), k, rho0, rho_p, rec, p, v);
    else
        store_record(i, rho_p[i], p, v, rec);
}

}  // namespace fg
