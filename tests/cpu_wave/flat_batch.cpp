// The flat density schedule of a batch over scenes of unlike grids, run on the
// CPU with the cell tables in otherwise unreadable memory: exits 0 when every
// lookup stayed in them and every density is that of its scene.
//   flat_batch CELLS,PARTICLES CELLS,PARTICLES ...   (cells per axis)
#include "wave64.hpp"

// the assembly of the row loops, which do not run here
#define asm(...) ((void)0)
#define volatile(...) ("")
#include "fg_batch.hip"
#undef asm
#undef volatile

#include <algorithm>
#include <cstdarg>
#include <random>

namespace fg {
State& state() {
    static State s;
    return s;
}
void set_error(int, const char* fmt, ...) {
    va_list a;
    va_start(a, fmt);
    std::vfprintf(stderr, fmt, a);
    va_end(a);
}
bool check_launch(const char*) { return true; }
void launch_fill_u32(uint32_t* p, uint32_t v, uint64_t n, hipStream_t) { std::fill(p, p + n, v); }
void note_nbr_format(const void*, uint32_t, bool) {}
bool nbr_has_runs(const void*, uint32_t) { return false; }
}  // namespace fg
extern "C" int fg_peek_error(void) { return FG_ERR_INVALID_ARGUMENT; }
extern "C" hipError_t hipGetDevice(int*) { return hipErrorNoDevice; }
extern "C" hipError_t hipDeviceGetAttribute(int*, hipDeviceAttribute_t, int) { return hipErrorNoDevice; }
extern "C" hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int*, const void*, int, size_t) { return hipErrorNoDevice; }

int main(int argc, char** argv) {
    constexpr float h = 0.05f;
    std::vector<fg_scene_desc> scenes;
    std::vector<uint32_t> scene_of, key;
    std::vector<float4> pos;
    uint32_t buckets = 0;
    std::mt19937 rng(7);
    for (int k = 1; k < argc; k++) {
        int cells, count;
        if (std::sscanf(argv[k], "%d,%d", &cells, &count) != 2) return 2;
        fg_scene_desc d{};
        d.common.bucket_size = {cells, cells, cells};
        d.common.cell_size = {h, h, h};
        d.common.kernel_radius = h;
        d.common.kernel_radius_squared = h * h;
        d.common.simulation_scale = 1.0f;
        d.kernels.kPoly6 = 1.0f;
        d.gasConstant = 1.0f;
        d.mass = 1e12f;
        d.keyBase = buckets;
        d.particleBegin = (uint32_t)pos.size();
        d.particleCount = (uint32_t)count;
        // particles in all of the box, corners included
        std::uniform_real_distribution<float> u(0.0f, cells * h);
        for (int q = 0; q < count; q++) pos.push_back(make_float4(u(rng), u(rng), u(rng), 1.0f));
        scene_of.insert(scene_of.end(), (size_t)count, (uint32_t)scenes.size());
        scenes.push_back(d);
        buckets += (uint32_t)(cells * cells * cells);
    }
    const uint32_t n = (uint32_t)pos.size(), ns = (uint32_t)scenes.size();
    key.resize(n);
    wave64::launch(fg::k_batch_hash, dim3((n + 255) / 256), dim3(256), scenes.data(), ns, scene_of.data(), pos.data(), key.data(), n);
    std::vector<uint32_t> order(n);
    for (uint32_t i = 0; i < n; i++) order[i] = i;
    std::stable_sort(order.begin(), order.end(), [&](uint32_t a, uint32_t b) { return key[a] < key[b]; });
    std::vector<float4> sp(n), sv(n, make_float4(0, 0, 0, 0));
    uint32_t *start = wave64::guarded(buckets), *end = wave64::guarded(buckets);
    std::fill(start, start + buckets, fg::kEmpty);
    for (uint32_t i = n; i-- > 0;) {
        sp[i] = pos[order[i]];
        start[key[order[i]]] = i;
    }
    for (uint32_t i = 0; i < n; i++) end[key[order[i]]] = i + 1;
    std::vector<unsigned long long> nbr(256 * (size_t)n + 4096);
    std::vector<float2> rho(n);
    fg::state().flat_density = true;
    for (int block : {64, 128, 256, 512}) {
        fg::state().sph_block = block;
        std::fill(rho.begin(), rho.end(), make_float2(0, 0));
        if (fg::batch_density(scenes.data(), ns, scene_of.data(), sp.data(), sv.data(), rho.data(), start, end, nbr.data(), n,
                              fg::WorkQueue{nullptr, 1, 0}) != FG_OK)
            return 3;
        for (uint32_t i = 0; i < n; i++) {
            double want = 0.0;
            for (uint32_t j = 0; j < n; j++) {
                if (scene_of[i] != scene_of[j]) continue;
                const double dx = sp[i].x - sp[j].x, dy = sp[i].y - sp[j].y, dz = sp[i].z - sp[j].z;
                const double t = (double)h * h - (dx * dx + dy * dy + dz * dz);
                if (t > 0.0) want += t * t * t;
            }
            want *= 1e12;
            if (!(std::fabs(rho[i].x - want) <= 1e-5 * want)) {
                std::printf("particle %u of scene %u: density %g, not %g\n", i, scene_of[i], rho[i].x, want);
                return 1;
            }
        }
    }
    std::printf("ok: %u particles of %u scenes\n", n, ns);
    return 0;
}
