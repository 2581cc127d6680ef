// fg_sph.hip -- SPH density, pressure/viscosity forces with penalty walls,
// and symplectic-Euler integration (the work of GPU_Kernels/K_FluidSim.cu and
// K_Boundaries_Walls.cu).
//
// Two arithmetic forms share the launchers:
//  * reference form (FG_MATH_REFERENCE, and always for FG_KEY_REF_XOR): one
//    lane per sorted particle walks the 27 stencil buckets exactly as
//    K_FluidSim.cu:46-79/127-205 do, with per-bucket partial sums and the
//    same per-pair expressions, contraction off;
//  * fast form (FG_MATH_FAST with FG_KEY_LINEAR): the three x-neighbour cells
//    of a stencil row are consecutive keys, so their particles form one
//    contiguous range of the sorted arrays; a row (or its end cells) is
//    skipped when its nearest point is farther than h; the pair loop keeps
//    only what depends on j (r^2 test, (h^2-r^2)^3 for density; 1/r, h-r and
//    1/rho_j for forces) and applies m*kPoly6, m/rho_i, kSpiky, kVisc*mu once.
//    The neighbour set and summation order within a row are those of the
//    reference; only rounding differs.
#include "fg_internal.hpp"
#include "fg_sph_fast.hpp"
#include "fg_sph_tile.hpp"
#include "fg_sph_mixed.hpp"

#include <mutex>
#include <unordered_map>

namespace fg {

constexpr int kSphThreads = 256;

// Lanes per particle of the reference-arithmetic kernels (k_density_ref,
// k_forces_ref).  Up to kRefSpreadMax particles eight lanes a particle fill
// the GPU and keep eight bucket walks in flight; above, one lane a particle
// already does, and the groups' adding up costs more than it gains.  Measured
// with the reference's hash (density / forces, us):
//   24,108 particles   1 lane 51 / 90     8 lanes 14 / 24    16 lanes 15 / 31
//   108,000            1 lane 60 / 141    8 lanes 51 / 92    16 lanes 49 / 109
//   250,880            1 lane 98 / 185    8 lanes 125 / 212  16 lanes 131 / 249
//   1,048,576          1 lane 358 / 593   8 lanes 647 / 970
constexpr uint32_t kRefLanes = 8;
constexpr uint32_t kRefSpreadMax = 163840;

// ---------------------------------------------------------------------------
// Reference-arithmetic kernels
// ---------------------------------------------------------------------------
#pragma clang fp contract(off)

// Bucket of stencil offset (x,y,z) for a particle at p; false when the LINEAR
// cell lies outside the grid.
template <int MODE>
__device__ __forceinline__ bool stencil_bucket(const float4& p, const CellXYZ& c, int x, int y, int z,
                                               const fg_common_fluid_params& cp, uint32_t nb, uint32_t& b) {
    if (MODE == FG_KEY_REF_XOR) {
        const float ox = cp.cell_size.x * (float)x, oy = cp.cell_size.y * (float)y, oz = cp.cell_size.z * (float)z;
        b = hash_ref_xor(p.x + ox, p.y + oy, p.z + oz, cp.cell_size.x, cp.cell_size.y, cp.cell_size.z, nb);
        return true;
    } else {
        const int cx = c.x + x, cy = c.y + y, cz = c.z + z;
        if (cx < 0 || cy < 0 || cz < 0 || cx >= cp.bucket_size.x || cy >= cp.bucket_size.y || cz >= cp.bucket_size.z)
            return false;
        b = linear_key(cx, cy, cz, cp);
        return true;
    }
}

// The reference form spreads a particle's 27 buckets over LP lanes: lane sub
// walks buckets sub, sub + LP, ... of the z, y, x stencil order, each into a
// sum of its own from zero, and after each round the group adds the round's
// sums in bucket order.  The 27 walks are chains of dependent loads (bucket
// range, then its particles); one lane per particle walks them one after
// another with most of the GPU idle below a few hundred thousand particles.
// Sums equal to zero are not added: the running sum starts at +0 and so is
// never -0 under round-to-nearest, and adding +0 or -0 changes no bit.
//
// A pair whose squared distance exceeds h^2 (1 + 2^-20) has a distance more
// than two units in the last place above h, so its rounded square root
// exceeds h as well: it is rejected without the square root (most of a
// bucket's particles are).
//
// Bound by latency in small fluids and by VALU issue in large ones: a fluid
// of 24,108 particles with hashed keys takes 14 (density) and 24 us (forces),
// where one lane a particle, a powf a pair and every particle's terms under
// one branch took 105 and 109; 1,048,576 particles take 358 and 593 us, then
// 972 and 1,115.
__device__ __forceinline__ float ref_cut(float h) { return rn_mul(rn_mul(h, h), 0x1.00001p+0f); }

// x^3 (powf(x, 3.0f) in the reference) by way of 64 bits: x * x is exact
// there, the cube is rounded to 53 bits and then to 24, just over half a unit
// in the last place.
__device__ __forceinline__ float ref_cube(float x) {
    const double d = (double)x;
    return (float)(d * d * d);
}

// Adds the group's sums of one round to `total`, in lane order.
template <uint32_t LP>
__device__ __forceinline__ void ref_add_round(float& total, float part) {
    const uint32_t first = __lane_id() & ~(LP - 1u);
    uint32_t m = (uint32_t)(__ballot(part != 0.0f) >> first) & ((1u << LP) - 1u);
    while (m) {
        const int src = (int)first + __ffs((int)m) - 1;
        m &= m - 1u;
        total = rn_add(total, __shfl(part, src));
    }
}
template <uint32_t LP>
__device__ __forceinline__ void ref_add_round(F3& total, F3 part) {
    const uint32_t first = __lane_id() & ~(LP - 1u);
    uint32_t m = (uint32_t)(__ballot(part.x != 0.0f || part.y != 0.0f || part.z != 0.0f) >> first) & ((1u << LP) - 1u);
    while (m) {
        const int src = (int)first + __ffs((int)m) - 1;
        m &= m - 1u;
        total = add(total, f3(__shfl(part.x, src), __shfl(part.y, src), __shfl(part.z, src)));
    }
}

// K_FluidSim.cu:210-254 with ProcessMassDensityGridD (:46-79), by groups of LP lanes
template <int MODE, uint32_t LP>
__global__ void __launch_bounds__(kSphThreads)
    k_density_ref(const float4* __restrict__ sp, float2* __restrict__ rho_p, const uint32_t* __restrict__ start,
                  const uint32_t* __restrict__ end, uint32_t n, float k, float rho0, float m,
                  fg_common_fluid_params cp, fg_kernels_cache kc) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x, i = t / LP, lane = t % LP;
    if (i >= n) return;  // the same for every lane of a group
    const float4 p = sp[i];
    if (!(p.w > 0.0f)) return;
    const float s = cp.simulation_scale, h = cp.kernel_radius, h2 = cp.kernel_radius_squared;
    const float mkp = m * kc.kPoly6, cut = ref_cut(h);
    const uint32_t nb = dev_num_buckets(cp);
    CellXYZ c{0, 0, 0};
    if (MODE == FG_KEY_LINEAR) c = linear_cell(p.x, p.y, p.z, cp);
    const F3 p1 = mul(xyz(p), s);
    float rho = 0.0f;
    for (uint32_t r0 = 0; r0 < 27u; r0 += LP) {
        const int q = (int)(r0 + lane);
        float part = 0.0f;
        uint32_t b;
        if (q < 27 && stencil_bucket<MODE>(p, c, q % 3 - 1, (q / 3) % 3 - 1, q / 9 - 1, cp, nb, b)) {
            const uint32_t s0 = start[b], e0 = end[b];
            const uint32_t e = s0 != kEmpty ? min(e0, n) : 0u;
            for (uint32_t j0 = s0; j0 < e; j0 += 4u) {
                float4 cand[4];
#pragma unroll
                for (uint32_t u = 0; u < 4u; u++) cand[u] = sp[min(j0 + u, e - 1u)];
#pragma unroll
                for (uint32_t u = 0; u < 4u; u++) {
                    const F3 d = sub(p1, mul(xyz(cand[u]), s));
                    const float r2 = dot(d, d);
                    if (j0 + u >= e || r2 > cut) continue;
                    const float l = rn_sqrt(r2);
                    if (l < h) part = part + mkp * ref_cube(h2 - (l * l));
                }
            }
        }
        ref_add_round<LP>(rho, part);
    }
    if (lane == 0u) rho_p[i] = make_float2(fmaxf(1.0f, rho), k * (rho - rho0));
}

// Each lane's sums of one of its four buckets.
struct RefPart {
    float x[64], y[64], z[64];
};

// What the pair terms of particle i read, and the terms of one neighbour
// (K_FluidSim.cu:85-172) added to `total`.
struct RefPair {
    F3 p1, v1;
    float2 dp1;
    const float4* __restrict__ sp;
    const float4* __restrict__ sv;
    const float2* __restrict__ rho_p;
    float s, h, cut, kSpiky, kVisc, mu;

    __device__ __forceinline__ void add_terms(F3& total, uint32_t j) const {
        const float2 dp2 = rho_p[j];
        const F3 v2 = xyz(sv[j]);
        const F3 diff = sub(p1, mul(xyz(sp[j]), s));
        const float l = rn_sqrt(dot(diff, diff));
        if (l > h) return;  // both terms are zero
        // SPHCalculatePressureForceD, K_FluidSim.cu:107-120
        const float rr = dp1.x * dp2.x;
        const float pp = (dp1.y + dp2.y) / rr;
        const float r = kSpiky * ((h - l) * (h - l));
        total = add(total, mul(mul(mul(divs(diff, l), r), pp), -1.0f));
        // SPHCalculateViscosityForceD, K_FluidSim.cu:85-102
        const float lap = kVisc * (h - l);
        total = add(total, f3(((v2.x - v1.x) / rr) * lap * mu, ((v2.y - v1.y) / rr) * lap * mu,
                              ((v2.z - v1.z) / rr) * lap * mu));
    }

    // Bits of the cnt (<= 32) particles from b0 that may be within h.
    __device__ __forceinline__ uint32_t near(uint32_t b0, uint32_t cnt) const {
        uint32_t bits = 0u;
        for (uint32_t k = 0; k < cnt; k += 4u) {
            float4 cand[4];
#pragma unroll
            for (uint32_t u = 0; u < 4u; u++) cand[u] = sp[b0 + min(k + u, cnt - 1u)];
#pragma unroll
            for (uint32_t u = 0; u < 4u; u++) {
                const F3 d = sub(p1, mul(xyz(cand[u]), s));
                bits |= k + u < cnt && !(dot(d, d) > cut) ? 1u << (k + u) : 0u;
            }
        }
        return bits;
    }

    // Sum over the particles [s0, e) of a bucket of any length.
    __device__ __forceinline__ F3 bucket(uint32_t i, uint32_t s0, uint32_t e) const {
        F3 total = f3(0.0f, 0.0f, 0.0f);
        for (uint32_t b0 = s0; b0 < e; b0 += 32u) {
            uint32_t w = near(b0, min(e - b0, 32u));
            if (i - b0 < 32u) w &= ~(1u << (i - b0));
            for (; w; w &= w - 1u) add_terms(total, b0 + (uint32_t)__builtin_ctz(w));
        }
        return total;
    }
};

// K_FluidSim.cu:260-309 (+ fused integrate when pout != nullptr); with
// COUPLED, K_FluidSim.cu:315-413.  By groups of LP lanes, as k_density_ref.
template <int MODE, bool COUPLED, uint32_t LP>
__global__ void __launch_bounds__(kSphThreads)
    k_forces_ref(const float4* __restrict__ sp, const float4* __restrict__ sv, const float2* __restrict__ rho_p,
                 const uint32_t* __restrict__ start, const uint32_t* __restrict__ end, float4* __restrict__ vout,
                 float4* __restrict__ pout, const uint32_t* __restrict__ id, uint32_t n, float m, float mu,
                 fg_common_fluid_params cp, fg_kernels_cache kc, Contacts bc) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x, i = t / LP, lane = t % LP;
    if (i >= n) return;  // the same for every lane of a group
    const float4 pos = sp[i];
    const float4 vel = sv[i];
    F3 a = f3(0.0f, 0.0f, 0.0f);
    if (pos.w > 0.0f) {
        const float2 dp1 = rho_p[i];
        const uint32_t nb = dev_num_buckets(cp);
        const float s = cp.simulation_scale, h = cp.kernel_radius;
        CellXYZ c{0, 0, 0};
        if (MODE == FG_KEY_LINEAR) c = linear_cell(pos.x, pos.y, pos.z, cp);
        const RefPair pair{mul(xyz(pos), s), xyz(vel), dp1, sp, sv, rho_p, s, h, ref_cut(h), kc.kSpikyGradient,
                           kc.kViscosityLaplacian, mu};
        F3 internal = f3(0.0f, 0.0f, 0.0f);
        for (uint32_t q = 0; LP == 1u && q < 27u; q++) {
            uint32_t b;
            if (!stencil_bucket<MODE>(pos, c, (int)q % 3 - 1, (int)(q / 3u) % 3 - 1, (int)q / 9 - 1, cp, nb, b)) continue;
            const uint32_t s0 = start[b], e0 = end[b];
            if (s0 != kEmpty) ref_add_round<LP>(internal, pair.bucket(i, s0, min(e0, n)));
        }
        if constexpr (LP > 1u) {
            static_assert(LP == 1u || 4u * LP >= 27u, "four buckets a lane hold the stencil");
            __shared__ RefPart s_part[kSphThreads / 64][4];
            RefPart* const part = s_part[threadIdx.x / 64];
            const uint32_t wl = threadIdx.x % 64;
            // Four buckets a lane: where none holds more than 16 particles,
            // their particles are tested into one mask and those that may be
            // within h walked as one list, with a sum for each bucket (a
            // wavefront waits for the longest list, not four times for the
            // longest bucket; 24,389 particles 30 us bucket by bucket, 24 us
            // so; 108,288 100 and 92).  One lane a particle walks bucket by
            // bucket: as lists of four buckets 1,048,576 particles took 983 us
            // against 594.
            uint32_t s0[4], cnt[4];
            bool large = false;
#pragma unroll
            for (uint32_t u = 0; u < 4u; u++) {
                const int q = (int)(u * LP + lane);
                s0[u] = cnt[u] = 0u;
                uint32_t b;
                if (q < 27 && stencil_bucket<MODE>(pos, c, q % 3 - 1, (q / 3) % 3 - 1, q / 9 - 1, cp, nb, b)) {
                    s0[u] = start[b];
                    const uint32_t e = min(end[b], n);
                    cnt[u] = s0[u] != kEmpty && s0[u] < e ? e - s0[u] : 0u;
                    large |= cnt[u] > 16u;
                }
            }
            uint64_t near = 0;
#pragma unroll
            for (uint32_t u = 0; u < 4u; u++) {
                part[u].x[wl] = part[u].y[wl] = part[u].z[wl] = 0.0f;
                if (!large) near |= (uint64_t)pair.near(s0[u], cnt[u]) << (16u * u);
                if (!large && i - s0[u] < cnt[u]) near &= ~(1ull << (16u * u + (i - s0[u])));
            }
            F3 sum = f3(0.0f, 0.0f, 0.0f);
            uint32_t bucket = 4u;
            for (; near; near &= near - 1u) {
                const uint32_t k = (uint32_t)__builtin_ctzll(near), u = k >> 4;
                if (u != bucket) sum = f3(0.0f, 0.0f, 0.0f);
                bucket = u;
                pair.add_terms(sum, (u < 2u ? (u == 0u ? s0[0] : s0[1]) : (u == 2u ? s0[2] : s0[3])) + (k & 15u));
                part[u].x[wl] = sum.x;
                part[u].y[wl] = sum.y;
                part[u].z[wl] = sum.z;
            }
            if (large) {
#pragma unroll 1
                for (uint32_t u = 0; u < 4u; u++) {
                    const uint32_t a = u < 2u ? (u == 0u ? s0[0] : s0[1]) : (u == 2u ? s0[2] : s0[3]);
                    const uint32_t m4 = u < 2u ? (u == 0u ? cnt[0] : cnt[1]) : (u == 2u ? cnt[2] : cnt[3]);
                    const F3 f = pair.bucket(i, a, a + m4);
                    part[u].x[wl] = f.x;
                    part[u].y[wl] = f.y;
                    part[u].z[wl] = f.z;
                }
            }
#pragma unroll
            for (uint32_t u = 0; u < 4u; u++)
                ref_add_round<LP>(internal, f3(part[u].x[wl], part[u].y[wl], part[u].z[wl]));
        }
        // the body contact (fluid_external) with its cells over the same lanes
        F3 ext = f3(0.0f, 0.0f, 0.0f);
        if (COUPLED && bc.coupled) {
            if constexpr (LP == kContactLanes) {
                __shared__ ContactWave s_contact[kSphThreads / 64];
                ContactWave& contact = s_contact[threadIdx.x / 64];
                if (bc.st.enabled) ext = add(ext, contact_cells(pos, vel, bc.st, lane, contact));
                if (bc.dyn.enabled) ext = add(ext, contact_cells(pos, vel, bc.dyn, lane, contact));
            } else
                ext = fluid_external(pos, vel, bc);
        }
        if (lane != 0u) return;
        a = finish_accel_ext(internal, m, pos, vel, cp, COUPLED && bc.coupled, ext);
    }
    if (lane == 0u) write_back(id[i], n, pos, vel, a, cp, vout, pout);
}

// K_FluidSim.cu:418-438
__global__ void __launch_bounds__(256) k_integrate(float4* __restrict__ pos, const float4* __restrict__ vel,
                                                   uint32_t n, float q) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 p = pos[i];
    if (p.w > 0.0f) {
        const float4 v = vel[i];
        pos[i] = make_float4(p.x + v.x * q, p.y + v.y * q, p.z + v.z * q, p.w + v.w * q);
    }
}

#pragma clang fp contract(fast)

// ---------------------------------------------------------------------------
// Fast LINEAR kernels (per-particle work in fg_sph_fast.hpp)
// ---------------------------------------------------------------------------

template <bool MASKS, int BS>
__global__ void __launch_bounds__(BS)
    k_density_fast(const float4* __restrict__ sp, const float4* __restrict__ sv, float2* __restrict__ rho_p,
                   const uint32_t* __restrict__ start,
                   const uint32_t* __restrict__ end, uint32_t n, float k, float rho0, float m,
                   fg_common_fluid_params cp, fg_kernels_cache kc, unsigned long long* __restrict__ masks) {
    __shared__ DensityStage s_stage[BS / 64];  // one LDS slice per wavefront (staged row loop)
    const uint32_t i = xcd_block(blockIdx.x, gridDim.x) * BS + threadIdx.x;
    if ((i & ~63u) >= n) return;  // whole wavefronts; lanes past the last particle take part idle
    density_particle<MASKS>(i, sp, sv, rho_p, start, end, n, k, rho0, m, cp, kc, 0u, masks, nullptr,
                            &s_stage[threadIdx.x / 64]);
}

// Flat schedule (row table in LDS); same results as k_density_fast<MASKS>.
template <bool MASKS, int BS>
__global__ void __launch_bounds__(BS)
    k_density_flat(const float4* __restrict__ sp, const float4* __restrict__ sv, float2* __restrict__ rho_p,
                   const uint32_t* __restrict__ start,
                   const uint32_t* __restrict__ end, uint32_t n, float k, float rho0, float m,
                   fg_common_fluid_params cp, fg_kernels_cache kc, unsigned long long* __restrict__ masks) {
    __shared__ FlatWave s_flat[BS / 64];
    const uint32_t i = xcd_block(blockIdx.x, gridDim.x) * BS + threadIdx.x;
    if ((i & ~63u) >= n) return;
    const FlatRanges fr{&s_flat[threadIdx.x / 64], true};
    density_particle<MASKS>(i, sp, sv, rho_p, start, end, n, k, rho0, m, cp, kc, 0u, masks, &fr);
}

template <bool MASKS, bool COUPLED, int BS>
__global__ void __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(7)))
    k_forces_fast(const float4* __restrict__ sp, const float4* __restrict__ sv, const float2* __restrict__ rho_p,
                  const uint32_t* __restrict__ start, const uint32_t* __restrict__ end, float4* __restrict__ vout,
                  float4* __restrict__ pout, const uint32_t* __restrict__ id, uint32_t n, float m, float mu,
                  fg_common_fluid_params cp, fg_kernels_cache kc, const unsigned long long* __restrict__ masks,
                  Contacts bc, int runs) {
    // one LDS slice of kStageRecs neighbour records per wavefront (staged row loop)
    __shared__ float4 s_stage[MASKS ? (BS / 64) * 2 * kStageRecs : 1];
    // without masks: a slice of records with their cells
    __shared__ ForceStage s_tested[MASKS ? 1 : BS / 64];
    const uint32_t i = xcd_block(blockIdx.x, gridDim.x) * BS + threadIdx.x;
    if ((i & ~63u) >= n) return;  // whole wavefronts; lanes past the last particle take part idle
    forces_particle<MASKS, COUPLED>(i, sp, sv, rho_p, start, end, vout, pout, id, n, m, mu, cp, kc, 0u, masks, bc,
                                    nullptr, nullptr,
                                    MASKS && runs ? s_stage + (threadIdx.x / 64) * 2 * kStageRecs : nullptr,
                                    MASKS ? nullptr : &s_tested[threadIdx.x / 64]);
}

// Flat schedule (row table in LDS); same results as k_forces_fast<true, COUPLED>.
// amdgpu_waves_per_eu(8): the coupled variant's two body-grid descriptors
// take scalar registers (106 SGPRs without the hint, occupancy 7).
template <bool COUPLED, int BS>
__global__ void __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(8)))
    k_forces_flat(const float4* __restrict__ sp, const float4* __restrict__ sv, const float2* __restrict__ rho_p,
                  const uint32_t* __restrict__ start, const uint32_t* __restrict__ end, float4* __restrict__ vout,
                  float4* __restrict__ pout, const uint32_t* __restrict__ id, uint32_t n, float m, float mu,
                  fg_common_fluid_params cp, fg_kernels_cache kc, const unsigned long long* __restrict__ masks,
                  Contacts bc) {
    __shared__ uint32_t s_rb[9 * BS];
    __shared__ uint32_t s_mm[9 * BS];
    const uint32_t i = xcd_block(blockIdx.x, gridDim.x) * BS + threadIdx.x;
    if (i >= n) return;
    FlatRows fr{s_rb, s_mm, (uint32_t)BS, (uint32_t)threadIdx.x};
    forces_particle<true, COUPLED>(i, sp, sv, rho_p, start, end, vout, pout, id, n, m, mu, cp, kc, 0u, masks, bc,
                                   &fr);
}

// The coupled masked force pass with body contact deferred: a particle
// inside a body grid's expanded bounds stores its pair sum and joins a list
// (forces_particle with DEFER); the others finish here without the contact
// walk, which leaves the wavefronts that never meet a body free of it.  The
// row loop is that of k_forces_fast<true, true>: each row's records staged in
// LDS a row ahead, at the runs that the density pass left (with `runs`).
template <int BS>
__global__ void __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(7)))
    k_forces_deferred(const float4* __restrict__ sp, const float4* __restrict__ sv, const float2* __restrict__ rho_p,
                      const uint32_t* __restrict__ start, const uint32_t* __restrict__ end,
                      float4* __restrict__ vout, float4* __restrict__ pout, const uint32_t* __restrict__ id,
                      uint32_t n, float m, float mu, fg_common_fluid_params cp, fg_kernels_cache kc,
                      const unsigned long long* __restrict__ masks, Contacts bc, DeferredContact dc, int runs) {
    __shared__ float4 s_stage[(BS / 64) * 2 * kStageRecs];
    const uint32_t i = xcd_block(blockIdx.x, gridDim.x) * BS + threadIdx.x;
    if ((i & ~63u) >= n) return;
    forces_particle<true, true, true>(i, sp, sv, rho_p, start, end, vout, pout, id, n, m, mu, cp, kc, 0u, masks,
                                   bc, nullptr, &dc, runs ? s_stage + (threadIdx.x / 64) * 2 * kStageRecs : nullptr);
}

// Second pass of the deferred form: body contact (fluid_external: the
// static grid, then the dynamic one, summed from zero), walls, clamp and
// integration of the listed particles from their pair sums.  Each particle
// takes a group of lanes that walk its body-grid cells together
// (contact_cells, bit-identical to the one-lane walk).  Six wavefronts a SIMD
// (80 registers, 16 bytes of scratch): 58 us, the compiler's five 64 us, at
// 1,048,576 particles of which 112k are listed.
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(6)))
    k_contact_finish(const float4* __restrict__ sp, const float4* __restrict__ sv, float4* __restrict__ vout,
                     float4* __restrict__ pout, const uint32_t* __restrict__ id, uint32_t n, float m,
                     fg_common_fluid_params cp, Contacts bc, DeferredContact dc) {
    __shared__ ContactWave s_contact[256 / 64];
    ContactWave& contact = s_contact[threadIdx.x / 64];
    const uint32_t cnt = min(*dc.count, n);
    const uint32_t sub = threadIdx.x % kContactLanes;
    const uint32_t groups = gridDim.x * (blockDim.x / kContactLanes);
    // k is the same on every lane of a group, so a group is active or idle as a whole
    for (uint32_t k = (blockIdx.x * blockDim.x + threadIdx.x) / kContactLanes; k < cnt; k += groups) {
        const uint32_t i = dc.list[k];
        const float4 pos = sp[i], vel = sv[i];
        F3 e = f3(0.0f, 0.0f, 0.0f);
        if (bc.st.enabled) e = add(e, contact_cells(pos, vel, bc.st, sub, contact));
        if (bc.dyn.enabled) e = add(e, contact_cells(pos, vel, bc.dyn, sub, contact));
        if (sub != 0) continue;
        const float4 ia = dc.acc[i];
        const F3 a = finish_accel_ext(f3(ia.x, ia.y, ia.z), m, pos, vel, cp, bc.coupled != 0, e);
        write_back(id[i], n, pos, vel, a, cp, vout, pout);
    }
}

// Mixed-precision density (fg_sph_mixed.hpp): the FP32 pass's masks and
// records, FP16-culled candidates, compensated sums.
template <int BS>
__global__ void __launch_bounds__(BS)
    k_density_mixed(const float4* __restrict__ sp, const float4* __restrict__ sv, float2* __restrict__ rho_p,
                    const uint32_t* __restrict__ start, const uint32_t* __restrict__ end, uint32_t n, float k,
                    float rho0, float m, fg_common_fluid_params cp, fg_kernels_cache kc,
                    unsigned long long* __restrict__ masks) {
    __shared__ MixedStage s_stage[BS / 64];
    const uint32_t i = xcd_block(blockIdx.x, gridDim.x) * BS + threadIdx.x;
    if ((i & ~63u) >= n) return;  // whole wavefronts; lanes past the last particle take part idle
    density_particle_mixed(i, sp, sv, rho_p, start, end, n, k, rho0, m, cp, kc, masks, s_stage[threadIdx.x / 64]);
}

// LDS-tiled passes (fg_sph_tile.hpp).  Tile b of the grid is the sorted
// particles [b * kTileLanes, (b + 1) * kTileLanes); blocks are remapped so
// each XCD walks a contiguous range of tiles.
__global__ void __launch_bounds__(kTileLanes)
    k_density_tile(const float4* __restrict__ sp, const float4* __restrict__ sv, float2* __restrict__ rho_p,
                   const uint32_t* __restrict__ start, const uint32_t* __restrict__ end, uint32_t n, float k,
                   float rho0, float m, fg_common_fluid_params cp, fg_kernels_cache kc,
                   unsigned long long* __restrict__ masks) {
    __shared__ TileGeom g;
    __shared__ TileSetupLds L;
    __shared__ float4 lpos[kTileCap];
    __shared__ __align__(16) uint16_t llists[kTileLanes * kListMax];
    const uint32_t tile = xcd_block(blockIdx.x, gridDim.x);
    const uint32_t i = tile * kTileLanes + threadIdx.x;
    const bool have = i < n;
    const uint32_t nvalid = min(n - tile * kTileLanes, (uint32_t)kTileLanes);
    const float4 p = have ? sp[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const float4 v = have ? sv[i] : p;  // (loaded before the set-up, whose latency it shares)
    const uint32_t fb = tile_setup(g, L, n, nvalid, have, p, cp, 0u, start, end);
    // the staging plan, for the force pass
    if (threadIdx.x < kTileDescWords) {
        const uint32_t t = threadIdx.x, nseg = fb ? 0u : 9u * g.nrows;
        uint32_t v = 0u;
        if (t == 0) v = fb;
        else if (t == 1) v = fb ? 0u : g.nrows;
        else if (t == 2) v = fb ? 0u : g.total;
        else if (t >= 4 && t < 4 + (uint32_t)kTileSegs) v = t - 4 < nseg ? g.sb[t - 4] : 0u;
        else if (t >= 4 + (uint32_t)kTileSegs && t < 4 + 2 * (uint32_t)kTileSegs)
            v = t - 4 - kTileSegs < nseg ? g.len[t - 4 - kTileSegs] : 0u;
        else if (t >= 4 + 2 * (uint32_t)kTileSegs && t < 4 + 3 * (uint32_t)kTileSegs)
            v = t - 4 - 2 * kTileSegs < nseg ? g.off[t - 4 - 2 * kTileSegs] : 0u;
        nbr_descs(masks, n)[(size_t)tile * kTileDescWords + t] = v;
    }
    if (fb) {
        if (have) {
            density_particle<true>(i, sp, sv, rho_p, start, end, n, k, rho0, m, cp, kc, 0u, masks);
            nbr_counts(masks, n)[i] = kListOverflow;
        }
        return;
    }
    tile_fill(g, sp, 1, lpos);
    tile_fill_wait();
    if (have)
        tile_density_particle(g, lpos, llists + threadIdx.x * kListMax, i, p, v, rho_p, start, end, n, k, rho0, m,
                              cp, kc, masks);
}

template <bool COUPLED>
__global__ void __launch_bounds__(kTileLanes)
    k_forces_tile(const float4* __restrict__ sp, const float4* __restrict__ sv, const float2* __restrict__ rho_p,
                  const uint32_t* __restrict__ start, const uint32_t* __restrict__ end, float4* __restrict__ vout,
                  float4* __restrict__ pout, const uint32_t* __restrict__ id, uint32_t n, float m, float mu,
                  fg_common_fluid_params cp, fg_kernels_cache kc, const unsigned long long* __restrict__ masks,
                  Contacts bc) {
    __shared__ TileGeom g;
    __shared__ __align__(16) float4 recs[2 * kTileCap];
    float4* recA = recs;
    float4* recB = recs + kTileCap;
    const uint32_t tile = xcd_block(blockIdx.x, gridDim.x);
    const uint32_t i = tile * kTileLanes + threadIdx.x;
    const bool have = i < n;
    // Everything a lane needs besides the staged records is loaded first, so
    // its latency overlaps the descriptor load and the staging.
    float4 pos = make_float4(0.0f, 0.0f, 0.0f, 0.0f), vel = pos;
    float2 dpi = make_float2(1.0f, 0.0f);
    uint32_t cnt = 0u, oid = n;
    uint4 l0 = make_uint4(0u, 0u, 0u, 0u), l1 = l0;
    if (have) {
        const uint4* lists = nbr_lists(masks, n);
        pos = sp[i];
        vel = sv[i];
        dpi = rho_p[i];
        cnt = nbr_counts(masks, n)[i];
        oid = id[i];
        l0 = lists[i];
        l1 = lists[(size_t)n + i];
    }
    // the staging plan the density pass wrote for this tile
    if (threadIdx.x < kTileDescWords) {
        const uint32_t t = threadIdx.x;
        const uint32_t v = nbr_descs(masks, n)[(size_t)tile * kTileDescWords + t];
        if (t == 0) g.fallback = v;
        else if (t == 1) g.nrows = v;
        else if (t == 2) g.total = v;
        else if (t >= 4 && t < 4 + (uint32_t)kTileSegs) g.sb[t - 4] = v;
        else if (t >= 4 + (uint32_t)kTileSegs && t < 4 + 2 * (uint32_t)kTileSegs) g.len[t - 4 - kTileSegs] = v;
        else if (t >= 4 + 2 * (uint32_t)kTileSegs && t < 4 + 3 * (uint32_t)kTileSegs)
            g.off[t - 4 - 2 * kTileSegs] = v;
    }
    __syncthreads();
    if (g.fallback != 0u || g.total > kTileCap || g.nrows > (uint32_t)kTileRowsMax) {
        if (have)
            forces_particle<true, COUPLED>(i, sp, sv, rho_p, start, end, vout, pout, id, n, m, mu, cp, kc, 0u, masks,
                                           bc);
        return;
    }
    const float4* rec = nbr_records(masks, n);
    tile_fill(g, rec, 2, recA);
    tile_fill(g, rec + 1, 2, recB);
    tile_fill_wait();
    if (!have) return;
    F3 a = f3(0.0f, 0.0f, 0.0f);
    if (pos.w > 0.0f) {
        if (cnt > kListMax) cnt = kListOverflow;  // (a count the density pass cannot write reads the masks)
        a = tile_forces_particle<COUPLED>(recA, recB, i, pos, vel, dpi, cnt, l0, l1, sp, sv, rho_p, start, end, n, m,
                                          mu, cp, kc, masks, bc);
    }
    write_back(oid, n, pos, vel, a, cp, vout, pout);
}

// ---------------------------------------------------------------------------
// Launch helpers
// ---------------------------------------------------------------------------

// Which form the last density pass wrote into a neighbour buffer, and for how
// many particles: lists (the tiled pass) or row masks with the wavefronts'
// runs.  The force pass follows it, whatever the schedule is when it runs, so
// the two passes always agree on the format; a buffer that no density pass of
// this process wrote for that many particles is read by its row masks alone.
struct NbrFormat {
    uint32_t n;
    bool tiled;
};
static std::mutex g_nbr_mu;
static std::unordered_map<const void*, NbrFormat>& nbr_formats() {
    static std::unordered_map<const void*, NbrFormat> m;
    return m;
}
void note_nbr_format(const void* masks, uint32_t n, bool tiled) {
    std::lock_guard<std::mutex> lock(g_nbr_mu);
    nbr_formats()[masks] = NbrFormat{n, tiled};
}
static bool nbr_format_tiled(const void* masks) {
    std::lock_guard<std::mutex> lock(g_nbr_mu);
    auto it = nbr_formats().find(masks);
    return it != nbr_formats().end() && it->second.tiled;
}
bool nbr_has_runs(const void* masks, uint32_t n) {
    std::lock_guard<std::mutex> lock(g_nbr_mu);
    auto it = nbr_formats().find(masks);
    return n >= kRunMinParticles && it != nbr_formats().end() && !it->second.tiled && it->second.n == n;
}
// Neighbour buffers whose FP16 pair records a cell pass has written, with
// the particle count it wrote them for (the records' place depends on it).
static std::unordered_map<const void*, uint32_t>& half_written() {
    static std::unordered_map<const void*, uint32_t> m;
    return m;
}
void note_half_records(const void* buf, uint32_t n) {
    std::lock_guard<std::mutex> lock(g_nbr_mu);
    half_written()[buf] = n;
}
static bool half_records_for(const void* buf, uint32_t n) {
    std::lock_guard<std::mutex> lock(g_nbr_mu);
    auto it = half_written().find(buf);
    return it != half_written().end() && it->second == n;
}
static bool have_params(const char* who) {
    if (!state().have_common || !state().have_kernels) {
        set_error(FG_ERR_NOT_INITIALIZED, "%s: call gInitializeCommonFluidParams and gInitializeKernelParams first",
                  who);
        return false;
    }
    return true;
}

// The density and force passes walk the 27 cells around a particle's own,
// which holds every neighbour only when the cells are at least h on every
// axis; smaller cells are refused rather than summed short.
static bool stencil_covers_h(const char* who) {
    const fg_common_fluid_params& cp = state().common;
    const float s = cp.simulation_scale;
    if (linear_reach(cp.kernel_radius, s, cp.cell_size.x) > 1 ||
        linear_reach(cp.kernel_radius, s, cp.cell_size.y) > 1 ||
        linear_reach(cp.kernel_radius, s, cp.cell_size.z) > 1) {
        set_error(FG_ERR_UNSUPPORTED, "%s: cell_size is smaller than the kernel radius (the 27-cell stencil "
                  "would miss neighbours)", who);
        return false;
    }
    return true;
}

static bool use_fast() { return state().key_mode == FG_KEY_LINEAR && state().math_mode == FG_MATH_FAST; }

#define FG_SPH_LAUNCH_BS(KERN, BS, n, ...) \
    hipLaunchKernelGGL(KERN, dim3(grid_for(n, BS)), dim3(BS), 0, state().stream, __VA_ARGS__)

// Launch KERN<A, BS> / KERN<A, B, BS> with BS = the tuned SPH block size.
#define FG_SPH_LAUNCH(KERN, A, n, ...)                                                                      \
    do {                                                                                                    \
        switch (state().sph_block) {                                                                        \
            case 64: FG_SPH_LAUNCH_BS((KERN<A, 64>), 64, n, __VA_ARGS__); break;                            \
            case 128: FG_SPH_LAUNCH_BS((KERN<A, 128>), 128, n, __VA_ARGS__); break;                         \
            case 512: FG_SPH_LAUNCH_BS((KERN<A, 512>), 512, n, __VA_ARGS__); break;                         \
            default: FG_SPH_LAUNCH_BS((KERN<A, 256>), 256, n, __VA_ARGS__);                                \
        }                                                                                                   \
    } while (0)

#define FG_SPH_LAUNCH2(KERN, A, B, n, ...)                                                                  \
    do {                                                                                                    \
        switch (state().sph_block) {                                                                        \
            case 64: FG_SPH_LAUNCH_BS((KERN<A, B, 64>), 64, n, __VA_ARGS__); break;                         \
            case 128: FG_SPH_LAUNCH_BS((KERN<A, B, 128>), 128, n, __VA_ARGS__); break;                      \
            case 512: FG_SPH_LAUNCH_BS((KERN<A, B, 512>), 512, n, __VA_ARGS__); break;                      \
            default: FG_SPH_LAUNCH_BS((KERN<A, B, 256>), 256, n, __VA_ARGS__);                             \
        }                                                                                                   \
    } while (0)

// Launch the reference form with kRefLanes lanes or one lane a particle.
#define FG_REF_LAUNCH(SPREAD, SINGLE, ...)                                                                            \
    do {                                                                                                              \
        if (n <= kRefSpreadMax)                                                                                       \
            hipLaunchKernelGGL(SPREAD, dim3(grid_for((uint64_t)n * kRefLanes, kSphThreads)), dim3(kSphThreads), 0,    \
                               st.stream, __VA_ARGS__);                                                               \
        else                                                                                                          \
            hipLaunchKernelGGL(SINGLE, dim3(grid_for(n, kSphThreads)), dim3(kSphThreads), 0, st.stream, __VA_ARGS__); \
    } while (0)

int launch_density(float4* sp, float2* rho_p, uint32_t* start, uint32_t* end, uint32_t n, float k, float rho0,
                   float m, unsigned long long* masks = nullptr, const float4* sv = nullptr) {
    if (!stencil_covers_h("density pass")) return FG_ERR_UNSUPPORTED;
    const State& st = state();
    const bool mixed = st.precision == FG_PRECISION_MIXED && use_fast() && masks;
    if (mixed && !half_records_for(masks, n)) {
        set_error(FG_ERR_NOT_INITIALIZED, "density pass (mixed precision): no cell pass has written FP16 offsets "
                  "for %u particles into this neighbour buffer (fg_cell_offsets_pos_vel with neighborBuffer)", n);
        return FG_ERR_NOT_INITIALIZED;
    }
    if (masks && use_fast()) note_nbr_format(masks, n, st.tiled && !mixed);
    if (mixed)
        FG_SPH_LAUNCH_BS(k_density_mixed<64>, 64, n, sp, sv, rho_p, start, end, n, k, rho0, m, st.common,
                         st.kernels, masks);
    else if (use_fast() && masks && st.tiled)
        hipLaunchKernelGGL(k_density_tile, dim3(grid_for(n, kTileLanes)), dim3(kTileLanes), 0, st.stream, sp, sv,
                           rho_p, start, end, n, k, rho0, m, st.common, st.kernels, masks);
    else if (use_fast() && masks && st.flat_density)
        FG_SPH_LAUNCH(k_density_flat, true, n, sp, sv, rho_p, start, end, n, k, rho0, m, st.common, st.kernels, masks);
    else if (use_fast() && masks)
        FG_SPH_LAUNCH(k_density_fast, true, n, sp, sv, rho_p, start, end, n, k, rho0, m, st.common, st.kernels, masks);
    else if (use_fast())
        FG_SPH_LAUNCH(k_density_fast, false, n, sp, (const float4*)nullptr, rho_p, start, end, n, k, rho0, m, st.common, st.kernels,
                      (unsigned long long*)nullptr);
    else if (st.key_mode == FG_KEY_LINEAR)
        FG_REF_LAUNCH((k_density_ref<FG_KEY_LINEAR, kRefLanes>), (k_density_ref<FG_KEY_LINEAR, 1>), sp, rho_p, start,
                      end, n, k, rho0, m, st.common, st.kernels);
    else
        FG_REF_LAUNCH((k_density_ref<FG_KEY_REF_XOR, kRefLanes>), (k_density_ref<FG_KEY_REF_XOR, 1>), sp, rho_p, start,
                      end, n, k, rho0, m, st.common, st.kernels);
    return check_launch("density") ? FG_OK : fg_peek_error();
}

int launch_forces(float4* sp, float4* sv, float2* rho_p, uint32_t* start, uint32_t* end, float4* vout,
                  float4* pout, uint32_t* id, uint32_t n, float m, float mu, const unsigned long long* masks = nullptr,
                  const Contacts* bcp = nullptr) {
    if (!stencil_covers_h("force pass")) return FG_ERR_UNSUPPORTED;
    Contacts bc{};
    if (bcp) bc = *bcp;
    const bool coupled = bc.coupled != 0;
    const State& st = state();
    if (use_fast() && masks && nbr_format_tiled(masks)) {
        if (coupled)
            hipLaunchKernelGGL(k_forces_tile<true>, dim3(grid_for(n, kTileLanes)), dim3(kTileLanes), 0, st.stream, sp,
                               sv, rho_p, start, end, vout, pout, id, n, m, mu, st.common, st.kernels, masks, bc);
        else
            hipLaunchKernelGGL(k_forces_tile<false>, dim3(grid_for(n, kTileLanes)), dim3(kTileLanes), 0, st.stream,
                               sp, sv, rho_p, start, end, vout, pout, id, n, m, mu, st.common, st.kernels, masks, bc);
    } else if (use_fast() && masks && st.flat_forces) {
        if (coupled)
            FG_SPH_LAUNCH(k_forces_flat, true, n, sp, sv, rho_p, start, end, vout, pout, id, n, m, mu, st.common,
                          st.kernels, masks, bc);
        else
            FG_SPH_LAUNCH(k_forces_flat, false, n, sp, sv, rho_p, start, end, vout, pout, id, n, m, mu, st.common,
                          st.kernels, masks, bc);
    } else if (use_fast()) {
        const unsigned long long* mk = masks;
        const int runs = mk && nbr_has_runs(mk, n) ? 1 : 0;
        if (coupled && mk && st.defer_contact) {
            // The deferred particles' pair sums and list live in the neighbour
            // buffer's list area (used otherwise only by the tiled passes) and
            // the count in its count area; the count is cleared by a kernel,
            // not a memset, so the step can be captured in a graph.
            char* base = reinterpret_cast<char*>(const_cast<unsigned long long*>(mk));
            DeferredContact dc{reinterpret_cast<float4*>(base + nbr_list_offset(n)),
                               reinterpret_cast<uint32_t*>(base + nbr_list_offset(n) + 16 * (size_t)n),
                               reinterpret_cast<uint32_t*>(base + nbr_count_offset(n))};
            launch_fill_u32(dc.count, 0u, 1, st.stream);
            switch (st.sph_block) {
                case 64: FG_SPH_LAUNCH_BS(k_forces_deferred<64>, 64, n, sp, sv, rho_p, start, end, vout, pout, id, n,
                                          m, mu, st.common, st.kernels, mk, bc, dc, runs); break;
                case 128: FG_SPH_LAUNCH_BS(k_forces_deferred<128>, 128, n, sp, sv, rho_p, start, end, vout, pout, id,
                                           n, m, mu, st.common, st.kernels, mk, bc, dc, runs); break;
                case 512: FG_SPH_LAUNCH_BS(k_forces_deferred<512>, 512, n, sp, sv, rho_p, start, end, vout, pout, id,
                                           n, m, mu, st.common, st.kernels, mk, bc, dc, runs); break;
                default: FG_SPH_LAUNCH_BS(k_forces_deferred<256>, 256, n, sp, sv, rho_p, start, end, vout, pout, id,
                                          n, m, mu, st.common, st.kernels, mk, bc, dc, runs);
            }
            // up to one group of lanes per particle (the count is known only on the device)
            unsigned blocks = grid_for((uint64_t)n * kContactLanes, 256);
            if (blocks > 8192) blocks = 8192;
            hipLaunchKernelGGL(k_contact_finish, dim3(blocks), dim3(256), 0, st.stream, sp, sv, vout, pout, id, n, m,
                               st.common, bc, dc);
        } else if (coupled && mk)
            FG_SPH_LAUNCH2(k_forces_fast, true, true, n, sp, sv, rho_p, start, end, vout, pout, id, n, m, mu,
                           st.common, st.kernels, mk, bc, runs);
        else if (coupled)
            FG_SPH_LAUNCH2(k_forces_fast, false, true, n, sp, sv, rho_p, start, end, vout, pout, id, n, m, mu,
                           st.common, st.kernels, mk, bc, runs);
        else if (mk)
            FG_SPH_LAUNCH2(k_forces_fast, true, false, n, sp, sv, rho_p, start, end, vout, pout, id, n, m, mu,
                           st.common, st.kernels, mk, bc, runs);
        else
            FG_SPH_LAUNCH2(k_forces_fast, false, false, n, sp, sv, rho_p, start, end, vout, pout, id, n, m, mu,
                           st.common, st.kernels, mk, bc, runs);
    } else if (st.key_mode == FG_KEY_LINEAR) {
        if (coupled)
            FG_REF_LAUNCH((k_forces_ref<FG_KEY_LINEAR, true, kRefLanes>), (k_forces_ref<FG_KEY_LINEAR, true, 1>), sp, sv,
                          rho_p, start, end, vout, pout, id, n, m, mu, st.common, st.kernels, bc);
        else
            FG_REF_LAUNCH((k_forces_ref<FG_KEY_LINEAR, false, kRefLanes>), (k_forces_ref<FG_KEY_LINEAR, false, 1>), sp, sv,
                          rho_p, start, end, vout, pout, id, n, m, mu, st.common, st.kernels, bc);
    } else {
        if (coupled)
            FG_REF_LAUNCH((k_forces_ref<FG_KEY_REF_XOR, true, kRefLanes>), (k_forces_ref<FG_KEY_REF_XOR, true, 1>), sp, sv,
                          rho_p, start, end, vout, pout, id, n, m, mu, st.common, st.kernels, bc);
        else
            FG_REF_LAUNCH((k_forces_ref<FG_KEY_REF_XOR, false, kRefLanes>), (k_forces_ref<FG_KEY_REF_XOR, false, 1>), sp, sv,
                          rho_p, start, end, vout, pout, id, n, m, mu, st.common, st.kernels, bc);
    }
    return check_launch("forces") ? FG_OK : fg_peek_error();
}

}  // namespace fg

using namespace fg;

extern "C" {

// K_FluidSim.cu:488-518
void gCalcMassDensity(fg_float4* orderedPositions, fg_float2* mass_pressure, unsigned int* hashTable,
                      unsigned int* gridStart, unsigned int* gridEnd, int numParticles, float gasConstant,
                      float restDensity, float mass) {
    (void)hashTable;
    if (numParticles <= 0) return;
    if (!have_params("gCalcMassDensity")) return;
    if (!orderedPositions || !mass_pressure || !gridStart || !gridEnd) {
        set_error(FG_ERR_INVALID_ARGUMENT, "gCalcMassDensity: null pointer");
        return;
    }
    launch_density(FG_F4(orderedPositions), FG_F2(mass_pressure), gridStart, gridEnd, (uint32_t)numParticles,
                   gasConstant, restDensity, mass);
}

// K_FluidSim.cu:527-566
void gSPHCalculateForces(fg_float4* orderedPositions, fg_float4* orderedVelocity, fg_float4* forces,
                         fg_float2* density_pressure, unsigned int* gridStart, unsigned int* gridEnd, fg_float4* vel,
                         unsigned int* particleId, unsigned int numParticles, float mass, float viscosity) {
    (void)forces;
    if (numParticles == 0) return;
    if (!have_params("gSPHCalculateForces")) return;
    if (!orderedPositions || !orderedVelocity || !density_pressure || !gridStart || !gridEnd || !vel ||
        !particleId) {
        set_error(FG_ERR_INVALID_ARGUMENT, "gSPHCalculateForces: null pointer");
        return;
    }
    if ((void*)vel == (void*)orderedVelocity) {
        set_error(FG_ERR_INVALID_ARGUMENT, "gSPHCalculateForces: vel must not alias orderedVelocity");
        return;
    }
    launch_forces(FG_F4(orderedPositions), FG_F4(orderedVelocity), FG_F2(density_pressure), gridStart, gridEnd,
                  FG_F4(vel), nullptr, particleId, numParticles, mass, viscosity);
}

// K_FluidSim.cu:571-586
void gSPHIntegrate(fg_float4* _in_sph_positions, fg_float4* _in_sph_velocity, fg_float4* _in_sph_forces,
                   unsigned int _in_num_particles, fg_float2* _in_density_press, unsigned int* _in_grid_start,
                   unsigned int* _in_grid_end) {
    (void)_in_sph_forces;
    (void)_in_density_press;
    (void)_in_grid_start;
    (void)_in_grid_end;
    if (_in_num_particles == 0) return;
    if (!have_params("gSPHIntegrate")) return;
    if (!_in_sph_positions || !_in_sph_velocity) {
        set_error(FG_ERR_INVALID_ARGUMENT, "gSPHIntegrate: null pointer");
        return;
    }
    const State& st = state();
    float q;
    {
#pragma clang fp contract(off)
        q = st.common.deltaTimeIntegration / st.common.simulation_scale;
    }
    hipLaunchKernelGGL(k_integrate, dim3(grid_for(_in_num_particles, 256)), dim3(256), 0, st.stream,
                       FG_F4(_in_sph_positions), FG_F4(_in_sph_velocity), _in_num_particles, q);
    check_launch("gSPHIntegrate");
}

int fg_sph_forces_integrate(fg_float4* orderedPositions, fg_float4* orderedVelocity, fg_float2* density_pressure,
                            unsigned int* gridStart, unsigned int* gridEnd, fg_float4* vel, fg_float4* pos,
                            unsigned int* particleId, unsigned int numParticles, float mass, float viscosity) {
    if (numParticles == 0) return FG_OK;
    if (!have_params("fg_sph_forces_integrate")) return FG_ERR_NOT_INITIALIZED;
    if (!orderedPositions || !orderedVelocity || !density_pressure || !gridStart || !gridEnd || !vel || !pos ||
        !particleId) {
        set_error(FG_ERR_INVALID_ARGUMENT, "fg_sph_forces_integrate: null pointer");
        return FG_ERR_INVALID_ARGUMENT;
    }
    return launch_forces(FG_F4(orderedPositions), FG_F4(orderedVelocity), FG_F2(density_pressure), gridStart, gridEnd,
                         FG_F4(vel), FG_F4(pos), particleId, numParticles, mass, viscosity);
}

size_t fg_neighbor_mask_bytes(unsigned int numParticles) {
    // 9 row masks, then (each from a 256-byte boundary) a 32-byte neighbour
    // record, a u16 list count and a list of kListMax u16 per particle
    return nbr_buffer_bytes(numParticles);
}

int fg_sph_density_nbr(fg_float4* orderedPositions, const fg_float4* orderedVelocity, fg_float2* mass_pressure,
                       unsigned int* gridStart,
                       unsigned int* gridEnd, unsigned long long* neighborMasks, unsigned int numParticles,
                       float gasConstant, float restDensity, float mass) {
    if (numParticles == 0) return FG_OK;
    if (!have_params("fg_sph_density_nbr")) return FG_ERR_NOT_INITIALIZED;
    if (!orderedPositions || !orderedVelocity || !mass_pressure || !gridStart || !gridEnd || !neighborMasks) {
        set_error(FG_ERR_INVALID_ARGUMENT, "fg_sph_density_nbr: null pointer");
        return FG_ERR_INVALID_ARGUMENT;
    }
    return launch_density(FG_F4(orderedPositions), FG_F2(mass_pressure), gridStart, gridEnd, numParticles,
                          gasConstant, restDensity, mass, neighborMasks,
                          reinterpret_cast<const float4*>(orderedVelocity));
}

int fg_sph_forces_integrate_nbr(fg_float4* orderedPositions, fg_float4* orderedVelocity,
                                fg_float2* density_pressure, unsigned int* gridStart, unsigned int* gridEnd,
                                const unsigned long long* neighborMasks, fg_float4* vel, fg_float4* pos,
                                unsigned int* particleId, unsigned int numParticles, float mass, float viscosity) {
    if (numParticles == 0) return FG_OK;
    if (!have_params("fg_sph_forces_integrate_nbr")) return FG_ERR_NOT_INITIALIZED;
    if (!orderedPositions || !orderedVelocity || !density_pressure || !gridStart || !gridEnd || !neighborMasks ||
        !vel || !particleId) {
        set_error(FG_ERR_INVALID_ARGUMENT, "fg_sph_forces_integrate_nbr: null pointer");
        return FG_ERR_INVALID_ARGUMENT;
    }
    return launch_forces(FG_F4(orderedPositions), FG_F4(orderedVelocity), FG_F2(density_pressure), gridStart, gridEnd,
                         FG_F4(vel), pos ? FG_F4(pos) : nullptr, particleId, numParticles, mass, viscosity,
                         neighborMasks);
}

}  // extern "C"
