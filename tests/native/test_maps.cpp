// Map creation on the host stand-in (the layout kernel as a host loop): see test_native_cpu.py for the cases.
#include <stdio.h>
#include <string>

#include "hip_on_host.h"

#include "pp_copy.hip"
#include "pp_host.hip"

namespace pp_beam {
hipError_t init_noalloc_scratch(int) { return hipSuccess; }
}
namespace pp_strict {
hipError_t launch_interleave(const MapParts& src, const MapDesc& d, int64_t cols, double* raw, hipStream_t) {
    for (int64_t c = 0; c < cols; ++c)
        for (int64_t k = 0; k < d.ng[2]; ++k)
            for (int e = 0; e < d.ncomp; ++e)
                raw[(c * d.ng[2] + k) * d.ncomp + e] = src.comp[e][c * d.n[2] + (k < d.n[2] ? k : 0)];
    return hipSuccess;
}
}  // namespace pp_strict

static std::vector<double> axis(int n) {
    std::vector<double> a(n);
    for (int k = 0; k < n; ++k) a[k] = k;
    return a;
}

// Values in several pieces: a map without coefficient tables fits beside 256 MiB, and every node has its values.
static void pieces() {
    const int n[3] = {13, 1021, 1601};
    const int64_t nodes = (int64_t)n[0] * n[1] * n[2];
    const std::vector<double> gx = axis(n[0]), gy = axis(n[1]), gz = axis(n[2]);
    std::vector<double> v(nodes + 2);
    for (int64_t k = 0; k < nodes + 2; ++k) v[k] = (double)(k % 1000003);
    const double* parts[3] = {v.data(), v.data() + 1, v.data() + 2};
    for (int periodic = 0; periodic < 2; ++periodic) {
        const int64_t ngz = n[2] + periodic;
        const size_t table = sizeof(double) * 3 * n[0] * n[1] * ngz;
        budget = used + table + ((size_t)256 << 20) + ((size_t)1 << 20);
        pp_map* m = nullptr;
        CHECK(pp_map_create_parts(parts, 0, 3, n[0], n[1], n[2], gx.data(), gy.data(), gz.data(), 0.0,
                                  PP_MAP_NO_COEF | (periodic ? PP_MAP_PERIODIC_Z : 0), &m) == PP_OK);
        for (int64_t c = 0; c < (int64_t)n[0] * n[1]; ++c)
            for (int64_t k = 0; k < ngz; ++k)
                for (int e = 0; e < 3; ++e)
                    CHECK(m->d.raw[(c * ngz + k) * 3 + e] == parts[e][c * n[2] + (k < n[2] ? k : 0)]);
        CHECK(pp_map_destroy(m) == PP_OK);
        CHECK(pp_release_staging() == PP_OK && used == 0);
    }
}

int main(int argc, char** argv) {
    CHECK(argc == 2 && pp_init(0) == PP_OK);
    const std::string w = argv[1];
    if (w == "pieces") pieces();
    else CHECK(!"unknown case");
    return 0;
}
