// The library on a device that has no memory for some of its scratch: this program defines hipMalloc
// and hipFree itself (the dynamic linker binds libfia.so's calls to them), keeps account of the device
// memory in use and refuses what it is told to refuse, by asking the runtime for more than any device
// has, so that the library sees the runtime's own failure.  Nothing is enqueued by a refused call.
//
//   memory_caller <dir> <nx> <ny> <nz> <cell_length> <dt>
// reads <dir>/{rho,u,v,w}.bin (float32) and steps the density with an xz split and WENO6:
//   free      nothing refused; prints the sizes asked for in order, writes <dir>/free.bin
//   deny S    every request of S bytes refused, for each size S of the free run (S_exact: S bytes with
//             room to grow, and the same without); if the step succeeds all the same its density is
//             written to <dir>/deny_S.bin; then once more, nothing refused
//   capped    the density step and a pressure projection through one context, and through two, on a
//             device of just the memory that both take without the z stencil tables
#include <dlfcn.h>

#include <cstdio>
#include <cstdlib>
#include <fstream>
#include <map>
#include <mutex>
#include <set>
#include <string>
#include <vector>

#include "../include/fia.h"

namespace {

std::mutex lock;
std::map<void *, size_t> live;
size_t in_use = 0, peak = 0, most = (size_t)-1;
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
    if (denied.count(n) || in_use + n > most) {
        ++refused;
        const int e = next(p, (size_t)1 << 60);
        return e ? e : 2;
    }
    const int e = next(p, n);
    if (e == 0) {
        live[*p] = n;
        in_use += n;
        if (in_use > peak) peak = in_use;
    }
    return e;
}
extern "C" int hipFree(void *p) {
    static const auto next = real<int (*)(void *)>("hipFree");
    const std::lock_guard<std::mutex> hold(lock);
    const auto at = live.find(p);
    if (at != live.end()) {
        in_use -= at->second;
        live.erase(at);
    }
    return next(p);
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
fia_status project(fia_ctx *c, std::vector<float> &p) {
    std::vector<float> a = u, b = v, d = w;
    p.assign((size_t)nx * ny * nz, 0.0f);
    fia_grid3d g = {nx, ny, nz, h, nullptr, a.data(), b.data(), d.data(), 0};
    int it = 0;
    double res = 0.0;
    return fia_pressure_project(c, &g, nullptr, p.data(), 0, 1e-6, 2000, &it, &res);
}

// the density step on one context, a projection on another (or the same): two statuses
void sequence(const char *name, bool two) {
    std::vector<float> q, p;
    refused = 0;
    peak = in_use;
    fia_ctx *a = context(), *b = two ? context() : a;
    const fia_status s = density(a, q);
    const size_t held = fia_ctx_device_bytes(a);
    const fia_status t = project(b, p);
    std::printf("%s %d %d bytes %zu %zu peak %zu refused %d\n", name, (int)s, (int)t, held, fia_ctx_device_bytes(a), peak,
                refused);
    std::fflush(stdout);
    write_bin(name, q);
    write_bin(std::string(name) + "_p", p);
    if (two) fia_ctx_destroy(b);
    fia_ctx_destroy(a);
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

    std::vector<std::set<size_t>> cases;
    for (size_t s : std::set<size_t>(sizes.begin(), sizes.end())) cases.push_back({s});
    // five buffers of doubles in a row: records asked for with room to grow, refused without it too
    for (size_t i = 0; i + 4 < sizes.size(); ++i) {
        const size_t n = sizes[i] / sizeof(double), exact = n - n / 9;
        if (sizes[i + 1] == sizes[i] && sizes[i + 2] == sizes[i] && sizes[i + 3] == sizes[i] && sizes[i + 4] == sizes[i] &&
            exact + exact / 8 == n)
            cases.push_back({sizes[i], exact * sizeof(double)});
    }
    for (const std::set<size_t> &set : cases) {
        const std::string name = std::to_string(*set.rbegin()) + (set.size() > 1 ? "_exact" : "");
        c = context();
        refused = 0;
        denied = set;
        const fia_status e = density(c, q);
        const size_t held = fia_ctx_device_bytes(c);
        denied.clear();
        if (e == FIA_OK) write_bin("deny_" + name, q);
        const int times = refused;
        const fia_status again = density(c, q);
        std::printf("deny %s refused %d status %d bytes %zu again %d\n", name.c_str(), times, (int)e, held, (int)again);
        std::fflush(stdout);
        write_bin("again_" + name, q);
        fia_ctx_destroy(c);
    }

    // 32 bytes an entry, nz + 5 entries a row
    const size_t row = 32 * ((size_t)nz + 5);
    const std::set<size_t> tables = {row * nx * ny, row * nx * (ny + 1)};
    for (const bool two : {false, true}) {
        denied = tables;
        sequence(two ? "two_lean" : "one_lean", two);
        denied.clear();
        most = peak;
        sequence(two ? "two_capped" : "one_capped", two);
        most = (size_t)-1;
    }
    return 0;
}
