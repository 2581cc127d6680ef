// fg_mesh.hip -- generalized winding numbers of a triangle mesh on a point
// lattice, the device half of sampling a mesh into the rigid-body sphere sets
// of the reference's body particle files (RigidBody.cpp:55-108 reads a file
// that names its source mesh; the files were made from meshes offline).
//
// w(p) = sum over triangles of Omega_t(p) / (4 pi), Omega_t the signed solid
// angle of triangle t seen from p (Van Oosterom & Strackee, IEEE Trans.
// Biomed. Eng. 30(2), 1983):
//   tan(Omega / 2) = a.(b x c) / (|a||b||c| + (a.b)|c| + (b.c)|a| + (c.a)|b|)
// with a, b, c the corners minus p.  w is 1 inside and 0 outside a closed,
// outward-oriented mesh and degrades gracefully for open or self-intersecting
// ones (Jacobson et al., SIGGRAPH 2013).
//
// Every lattice point is independent and reads every triangle, an all-pairs
// shape.  The wavefronts of a workgroup share 64 * kMeshPts lattice points,
// kMeshPts neighbours of a row a lane, and a tile of triangles staged in LDS;
// each takes every WAVES-th triangle of the tile (LDS broadcasts), and the
// wavefronts' sums are added at the end, so a lattice of few points fills the
// chip too.  The per-point sums are FP64, so adding thousands of terms adds no
// error of its own.
//
// The work is bound by the instructions of a pair.  For most of them the
// triangle is small and far: with the triangle's normal n = (b - a) x (c - a)
// staged beside its corners the numerator is a.n (and free of the
// cancellation of a.(b x c)), and where it is under 1/8 of a denominator of
// positive terms the arc tangent is three terms of its series, 7e-9 of the
// value at most from the whole, with 1-ulp roots and reciprocal (about 40
// instructions a pair).  Other pairs, next to the surface, take exact roots,
// the numerator from the corners and atan2f.  20,000 triangles on 259,308
// points: 16.1 ms when every pair took the long way on its own, 4.9 ms so; on
// 12,716 points 12.0 and 0.75 ms.  Mean error against 64 bits on lattices
// through and around a mesh: 200 triangles 9.3e-9 the long way and 8.3e-9 so,
// 2,400 triangles 8.2e-9 and 2.4e-9.
//
// Of few triangles, large beside the lattice, most wavefronts have a near pair
// among each triangle's, and the short way before it is work on top: up to
// kMeshNearTris every pair takes the long way, four wavefronts a workgroup
// (their sums cost more than the pairs with sixteen).  On 8,000,000 points,
// both ways of a pair in sixteen wavefronts against the long way in four: 12
// triangles 483 and 240 us, 32 604 and 577, 64 832 and 1,115, 200 1,716 and
// 3,411.  The rule lies above where the times cross, where the errors do: the
// 1-ulp roots of pairs at under 1/8 add up to more than exact ones where there
// are few others (mean error of a 12-triangle box 3.5e-8 the long way; with
// 1-ulp roots throughout 5.1e-8).
#include "fg_internal.hpp"

namespace fg {

// Points a lane, and wavefronts a workgroup of many triangles.  20,000 triangles
// on 259,308 and on 12,716 points: 2 and 16 4.86 and 0.75 ms; 2 and 8 5.01 and 0.94; 3 and 16
// 5.09 and 1.00; 4 and 16 5.54 and 1.29; one point a lane 10.9 and 0.84 (LDS
// reads).
constexpr int kMeshPts = 2;
constexpr int kMeshWaves = 16, kMeshNearWaves = 4;
constexpr uint32_t kMeshNearTris = 128;
static_assert(kMeshNearWaves >= kMeshPts, "a wavefront for each of a lane's points adds the sums");
// Workgroups along x: a launch has fewer than 2^32 lanes in each dimension, so
// a lattice of more groups of points (268,435,456 points; half of that where
// they lie one to a row) goes on along y.
constexpr uint64_t kMeshMaxX = 1ull << 21;
static_assert(kMeshMaxX * 64 * kMeshWaves < (1ull << 32), "lanes along x");

#pragma clang fp contract(off)
// Lattice point (ix, iy, iz): origin + i * spacing per axis, product and sum
// each rounded to FP32.
__device__ __forceinline__ float3 mesh_lattice_point(fg_float3 o, float s, uint32_t ix, uint32_t iy, uint32_t iz) {
    return make_float3(o.x + (float)ix * s, o.y + (float)iy * s, o.z + (float)iz * s);
}
#pragma clang fp contract(fast)

// One triangle's half solid angle seen from (px, py, pz), the long way.
__device__ __forceinline__ float half_solid_angle_near(float px, float py, float pz, float4 v0, float4 v1, float4 v2) {
    const float ax = v0.x - px, ay = v0.y - py, az = v0.z - pz;
    const float bx = v1.x - px, by = v1.y - py, bz = v1.z - pz;
    const float cx = v2.x - px, cy = v2.y - py, cz = v2.z - pz;
    const float la = sqrtf(ax * ax + ay * ay + az * az);
    const float lb = sqrtf(bx * bx + by * by + bz * bz);
    const float lc = sqrtf(cx * cx + cy * cy + cz * cz);
    const float det = ax * (by * cz - bz * cy) + ay * (bz * cx - bx * cz) + az * (bx * cy - by * cx);
    const float den = la * lb * lc + (ax * bx + ay * by + az * bz) * lc + (bx * cx + by * cy + bz * cz) * la +
                      (cx * ax + cy * ay + cz * az) * lb;
    return atan2f(det, den);
}

// The same, the short way where the triangle is far; (v0.w, v1.w, v2.w) is its
// normal.  The x terms come last in every sum, so points that share py and pz
// share the rest.
__device__ __forceinline__ float half_solid_angle(float px, float py, float pz, float4 v0, float4 v1, float4 v2) {
    const float ax = v0.x - px, ay = v0.y - py, az = v0.z - pz;
    const float bx = v1.x - px, by = v1.y - py, bz = v1.z - pz;
    const float cx = v2.x - px, cy = v2.y - py, cz = v2.z - pz;
    const float a2 = __fmaf_rn(ax, ax, ay * ay + az * az), b2 = __fmaf_rn(bx, bx, by * by + bz * bz);
    const float c2 = __fmaf_rn(cx, cx, cy * cy + cz * cz);
    const float ab = __fmaf_rn(ax, bx, ay * by + az * bz), bc = __fmaf_rn(bx, cx, by * cy + bz * cz);
    const float ca = __fmaf_rn(cx, ax, cy * ay + cz * az);
    auto denominator = [&](float la, float lb, float lc) {
        return __fmaf_rn(ca, lb, __fmaf_rn(bc, la, __fmaf_rn(la, lb, ab) * lc));
    };
    const float den = denominator(__builtin_amdgcn_sqrtf(a2), __builtin_amdgcn_sqrtf(b2), __builtin_amdgcn_sqrtf(c2));
    const float num = __fmaf_rn(ax, v0.w, ay * v1.w + az * v2.w);
    // A denominator of positive terms, so that a root's ulp is no more of it;
    // above 1e-30 with each product above 1e-20, and with a reciprocal in range
    // (a NaN fails the tests).
    if (fminf(fminf(ab, bc), ca) > 1e-20f && fabsf(num) < 0.125f * den && den < 1e30f) {
        const float t = num * __builtin_amdgcn_rcpf(den), t2 = t * t;
        return t + t * t2 * (t2 * (0.2f - t2 * (1.0f / 7.0f)) - (1.0f / 3.0f));
    }
    const float det = ax * (by * cz - bz * cy) + ay * (bz * cx - bx * cz) + az * (bx * cy - by * cx);
    return atan2f(det, denominator(sqrtf(a2), sqrtf(b2), sqrtf(c2)));
}

template <int WAVES, bool SHORT>
__global__ void __launch_bounds__(64 * WAVES)
    k_mesh_winding(const fg_float3* __restrict__ verts, uint32_t nverts, const uint32_t* __restrict__ tris,
                   uint32_t ntris, fg_float3 origin, float spacing, uint32_t nx, uint32_t ny, uint32_t nz,
                   float* __restrict__ out) {
    constexpr int kTile = 64 * WAVES;
    __shared__ union {
        float4 tile[3][kTile];
        double sum[WAVES][64 * kMeshPts];
    } s;
    __shared__ uint32_t s_count[WAVES];
    const uint32_t lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    // the lane's points: kMeshPts neighbours in x, of one row of the lattice
    const uint32_t row_groups = nx / kMeshPts + (nx % kMeshPts != 0);
    const uint64_t first = ((uint64_t)blockIdx.y * gridDim.x + blockIdx.x) * 64;
    if (first >= (uint64_t)row_groups * ny * nz) return;  // past the lattice, the whole workgroup
    const uint64_t g = first + lane, row = g / row_groups;
    const uint32_t ix = (uint32_t)(g % row_groups) * kMeshPts;
    const float3 p0 = mesh_lattice_point(origin, spacing, ix, (uint32_t)(row % ny), (uint32_t)(row / ny));
    float px[kMeshPts];
    double acc[kMeshPts];
#pragma unroll
    for (int k = 0; k < kMeshPts; k++) {
        px[k] = mesh_lattice_point(origin, spacing, ix + k, 0, 0).x;
        acc[k] = 0.0;
    }
    for (uint64_t t0 = 0; t0 < ntris; t0 += kTile) {
        const uint64_t t = t0 + threadIdx.x;
        // A triangle naming a vertex that does not exist is left out.
        uint32_t i0 = nverts, i1 = nverts, i2 = nverts;
        if (t < ntris) {
            i0 = tris[3 * t];
            i1 = tris[3 * t + 1];
            i2 = tris[3 * t + 2];
        }
        const bool valid = i0 < nverts && i1 < nverts && i2 < nverts;
        const uint64_t lanes = __ballot(valid);
        __syncthreads();  // the previous tile has been read by every lane
        if (lane == 0) s_count[wave] = (uint32_t)__popcll(lanes);
        __syncthreads();
        uint32_t at = (uint32_t)__popcll(lanes & ((1ull << lane) - 1ull)), cnt = 0;
        for (uint32_t w = 0; w < (uint32_t)WAVES; w++) {
            if (w == wave) at += cnt;
            cnt += s_count[w];
        }
        if (valid) {
            const fg_float3 a = verts[i0], b = verts[i1], c = verts[i2];
            const double ux = (double)b.x - a.x, uy = (double)b.y - a.y, uz = (double)b.z - a.z;
            const double wx = (double)c.x - a.x, wy = (double)c.y - a.y, wz = (double)c.z - a.z;
            s.tile[0][at] = make_float4(a.x, a.y, a.z, (float)(uy * wz - uz * wy));
            s.tile[1][at] = make_float4(b.x, b.y, b.z, (float)(uz * wx - ux * wz));
            s.tile[2][at] = make_float4(c.x, c.y, c.z, (float)(ux * wy - uy * wx));
        }
        __syncthreads();
        for (uint32_t j = wave; j < cnt; j += WAVES) {
            const float4 v0 = s.tile[0][j], v1 = s.tile[1][j], v2 = s.tile[2][j];
#pragma unroll
            for (int k = 0; k < kMeshPts; k++)
                acc[k] += (double)(SHORT ? half_solid_angle(px[k], p0.y, p0.z, v0, v1, v2)
                                         : half_solid_angle_near(px[k], p0.y, p0.z, v0, v1, v2));
        }
    }
    // w = sum(2 atan2) / (4 pi)
    constexpr double kInv2Pi = 0.15915494309189533577;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kMeshPts; k++) s.sum[wave][k * 64 + lane] = acc[k];
    __syncthreads();
    if (wave >= (uint32_t)kMeshPts || row >= (uint64_t)ny * nz || ix + wave >= nx) return;
    double a = 0.0;  // wavefront k adds the sums of every lane's point k
    for (uint32_t w = 0; w < (uint32_t)WAVES; w++) a += s.sum[w][threadIdx.x];
    out[row * nx + ix + wave] = (float)(a * kInv2Pi);
}

}  // namespace fg

using namespace fg;

extern "C" {

int fg_mesh_winding_lattice(const fg_float3* vertices, unsigned int numVertices, const unsigned int* triangles,
                            unsigned int numTriangles, fg_float3 origin, float spacing, unsigned int nx,
                            unsigned int ny, unsigned int nz, float* winding) {
    const uint64_t npts = (uint64_t)nx * ny * nz;
    if (npts == 0) return FG_OK;
    if (!winding || (numTriangles && (!vertices || !triangles))) {
        set_error(FG_ERR_INVALID_ARGUMENT, "fg_mesh_winding_lattice: null pointer");
        return FG_ERR_INVALID_ARGUMENT;
    }
    if (!(spacing > 0.0f) || npts > (1ull << 34)) {
        set_error(FG_ERR_INVALID_ARGUMENT, "fg_mesh_winding_lattice: non-positive spacing or more than 2^34 points");
        return FG_ERR_INVALID_ARGUMENT;
    }
    const State& st = state();
    const uint64_t groups = (uint64_t)(nx / kMeshPts + (nx % kMeshPts != 0)) * ny * nz;
    const uint64_t blocks = (groups + 63) / 64, x = blocks < kMeshMaxX ? blocks : kMeshMaxX;
    const bool near = numTriangles <= kMeshNearTris;
    hipLaunchKernelGGL((near ? k_mesh_winding<kMeshNearWaves, false> : k_mesh_winding<kMeshWaves, true>),
                       dim3((unsigned)x, (unsigned)((blocks + x - 1) / x)), dim3(64 * (near ? kMeshNearWaves : kMeshWaves)),
                       0, st.stream, vertices, numVertices, triangles, numTriangles, origin, spacing, nx, ny, nz, winding);
    return check_launch("fg_mesh_winding_lattice") ? FG_OK : fg_peek_error();
}

}  // extern "C"
