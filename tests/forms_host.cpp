// Host side of the forms that the launchers of flux-interpolated-advection_amd/csrc/fia_kernels.hip
// choose by size and rule, built by tests/test_forms_host.py with hipcc; only the host code runs.
#include "pass_host.cpp"

// x planes per thread of the zero-velocity march on an nx x ny x nz cell grid, `block` threads a block
extern "C" long forms_zero_chunk(int nx, int ny, int nz, int block) {
    CompGrid g;
    g.init(-1, nx, ny, nz);
    return (long)zero_velocity_chunk(g, block);
}
