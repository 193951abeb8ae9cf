// The library on a device that has no memory for some of its scratch: this program defines hipMalloc
// itself (the dynamic linker binds libfia.so's calls to it) and refuses what it is told to refuse, by
// asking the runtime for more than any device has, so that the library sees the runtime's own failure.
//
//   memory_caller <dir> <nx> <ny> <nz> <cell_length> <dt>
// reads <dir>/{rho,u,v,w}.bin (float32) and steps the density with an xz split and WENO6:
//   free      nothing refused; prints the sizes asked for in order, writes <dir>/free.bin
//   deny S    every request of S bytes refused, for each size S of the free run; if the step succeeds
//             all the same its density is written to <dir>/deny_S.bin; then once more, nothing refused
#include <dlfcn.h>

#include <cstdio>
#include <cstdlib>
#include <fstream>
#include <mutex>
#include <set>
#include <string>
#include <vector>

#include "../include/fia.h"

namespace {

std::mutex lock;
int refused = 0;
std::vector<size_t> asked;
std::set<size_t> denied;

template <class F> F real(const char *name) {
    void *f = dlsym(RTLD_NEXT, name);
    if (!f) {
        std::fprintf(stderr, "no %s\n", name);
        std::exit(2);
    }
    return (F)f;
}

}  // namespace

extern "C" int hipMalloc(void **p, size_t n) {
    static const auto next = real<int (*)(void **, size_t)>("hipMalloc");
    const std::lock_guard<std::mutex> hold(lock);
    asked.push_back(n);
    if (denied.count(n)) {
        ++refused;
        const int e = next(p, (size_t)1 << 60);
        return e ? e : 2;
    }
    return next(p, n);
}

namespace {

int nx, ny, nz;
double h, dt;
std::string dir;
std::vector<float> rho, u, v, w;

std::vector<float> read_bin(const char *name, size_t n) {
    std::vector<float> a(n);
    std::ifstream f(dir + "/" + name + ".bin", std::ios::binary);
    f.read((char *)a.data(), (std::streamsize)(n * sizeof(float)));
    if (!f) {
        std::fprintf(stderr, "cannot read %s\n", name);
        std::exit(2);
    }
    return a;
}
void write_bin(const std::string &name, const std::vector<float> &a) {
    std::ofstream f(dir + "/" + name + ".bin", std::ios::binary);
    f.write((const char *)a.data(), (std::streamsize)(a.size() * sizeof(float)));
}

fia_ctx *context() {
    fia_ctx *c = nullptr;
    if (fia_ctx_create(0, &c) != FIA_OK) {
        std::fprintf(stderr, "%s\n", fia_last_error());
        std::exit(2);
    }
    return c;
}
fia_status density(fia_ctx *c, std::vector<float> &out) {
    out = rho;
    std::vector<float> a = u, b = v, d = w;
    fia_grid3d g = {nx, ny, nz, h, out.data(), a.data(), b.data(), d.data(), 0};
    fia_advect_opts o;
    fia_default_opts(&o);
    o.split_method = FIA_SPLIT_XZ_CELLFACE;
    return fia_move_substances_3d(c, &g, 0, dt, &o);
}
}  // namespace

int main(int argc, char **argv) {
    if (argc != 7) return 2;
    dir = argv[1];
    nx = std::atoi(argv[2]); ny = std::atoi(argv[3]); nz = std::atoi(argv[4]);
    h = std::atof(argv[5]); dt = std::atof(argv[6]);
    rho = read_bin("rho", (size_t)nx * ny * nz);
    u = read_bin("u", (size_t)(nx + 1) * ny * nz);
    v = read_bin("v", (size_t)nx * (ny + 1) * nz);
    w = read_bin("w", (size_t)nx * ny * (nz + 1));

    std::vector<float> q;
    fia_ctx *c = context();
    asked.clear();
    const fia_status first = density(c, q);
    const std::vector<size_t> sizes = asked;
    std::printf("free %d bytes %zu\nasked", (int)first, fia_ctx_device_bytes(c));
    for (size_t s : sizes) std::printf(" %zu", s);
    std::printf("\n");
    std::fflush(stdout);
    write_bin("free", q);
    fia_ctx_destroy(c);

    std::set<size_t> distinct(sizes.begin(), sizes.end());
    for (size_t s : distinct) {
        c = context();
        refused = 0;
        denied = {s};
        const fia_status e = density(c, q);
        const size_t held = fia_ctx_device_bytes(c);
        denied.clear();
        if (e == FIA_OK) write_bin("deny_" + std::to_string(s), q);
        const int times = refused;
        const fia_status again = density(c, q);
        std::printf("deny %zu refused %d status %d bytes %zu again %d\n", s, times, (int)e, held, (int)again);
        std::fflush(stdout);
        write_bin("again_" + std::to_string(s), q);
        fia_ctx_destroy(c);
    }
    return 0;
}
