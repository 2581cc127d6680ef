// The launch of fg_mesh_winding_lattice for a lattice of NX x NY x NZ points:
// prints the grid's x and y and the workgroup's lanes.
#include "wave64.hpp"

#include "fg_mesh.hip"

namespace fg {
State& state() {
    static State s;
    return s;
}
void set_error(int, const char*, ...) {}
bool check_launch(const char*) { return true; }
}  // namespace fg
extern "C" int fg_peek_error(void) { return FG_ERR_INVALID_ARGUMENT; }

int main(int argc, char** argv) {
    if (argc != 4) return 2;
    wave64::execute = false;
    const fg_float3 v[3] = {};
    const unsigned t[3] = {0, 1, 2};
    float out[1];
    const int rc = fg_mesh_winding_lattice(v, 3, t, 1, {0, 0, 0}, 1.0f, (unsigned)std::atol(argv[1]),
                                           (unsigned)std::atol(argv[2]), (unsigned)std::atol(argv[3]), out);
    if (rc != FG_OK || wave64::launches != 1) return 1;
    std::printf("%u %u %u\n", wave64::last_grid.x, wave64::last_grid.y, wave64::last_block.x);
    return 0;
}
