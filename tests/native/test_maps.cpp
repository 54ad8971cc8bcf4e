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
hipError_t launch_push_sum(int, const PushParams&, const SumParams&, int, hipStream_t) { return hipSuccess; }
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

// The layout of small maps, made on the host, is the kernel's: one table on either side of the line, both z forms.
static void layout() {
    for (int nz : {5, 6, 60, 70})
        for (int ncomp : {1, 3, 6})
            for (int periodic = 0; periodic < 2; ++periodic) {
                const int n[3] = {4, 5, nz};
                const int64_t ngz = nz + periodic;
                const std::vector<double> gx = axis(n[0]), gy = axis(n[1]), gz = axis(nz);
                std::vector<double> v((size_t)n[0] * n[1] * nz * ncomp);
                for (size_t k = 0; k < v.size(); ++k) v[k] = (double)k;
                pp_map* m = nullptr;
                CHECK(pp_map_create(v.data(), ncomp, n[0], n[1], nz, gx.data(), gy.data(), gz.data(), 0.0,
                                    PP_MAP_NO_COEF | (periodic ? PP_MAP_PERIODIC_Z : 0), &m) == PP_OK);
                for (int64_t c = 0; c < (int64_t)n[0] * n[1]; ++c)
                    for (int64_t k = 0; k < ngz; ++k)
                        for (int e = 0; e < ncomp; ++e)
                            CHECK(m->d.raw[(c * ngz + k) * ncomp + e] ==
                                  v[(size_t)(((int64_t)e * n[0] * n[1] + c) * nz + (k < nz ? k : 0))]);
                CHECK(pp_map_destroy(m) == PP_OK);
            }
}

// A term may share the cell lookup of the map before it only if every node is the same.
static void same_cell() {
    std::vector<double> gx = {0, 1, 2.5, 4}, zx = {-0.0, 1, 2.5, 4}, hx = {0, 1.25, 2.5, 4}, one = {0}, v(4, 1.0);
    const double* parts[3] = {v.data(), v.data(), v.data()};
    auto make = [&](const std::vector<double>& g) {
        pp_map* m = nullptr;
        CHECK(pp_map_create_parts(parts, 0, 3, 1, 1, (int)g.size(), one.data(), one.data(), g.data(), 0.0, PP_MAP_NO_COEF,
                                  &m) == PP_OK);
        return m;
    };
    pp_map *a = make(gx), *twin = make(zx), *b = make(hx);
    double state[6] = {};
    pp_push_args args;
    memset(&args, 0, sizeof(args));
    args.algorithm = PP_ALG_BORIS;
    args.precision = PP_PREC_FP64;
    args.n = args.nsteps = 1;
    args.x = state; args.y = state + 1; args.z = state + 2;
    args.vx = state + 3; args.vy = state + 4; args.vz = state + 5;
    pp_sum_term t[3];
    memset(t, 0, sizeof(t));
    for (auto& q : t) {
        q.field.kind = PP_FIELD_MAP;
        q.field.scale1 = q.weight = 1.0;
    }
    t[1].flags = PP_SUM_SAME_CELL;
    t[0].field.map = a;
    t[1].field.map = twin;
    CHECK(pp_push_sum(&args, t, 2, nullptr) == PP_OK);
    t[1].field.map = a;
    CHECK(pp_push_sum(&args, t, 2, nullptr) == PP_OK);
    t[1].field.map = b;                                     // same count and ends, another node inside
    CHECK(pp_push_sum(&args, t, 2, nullptr) == PP_ERR_INVALID);
    t[1].flags = 0;
    CHECK(pp_push_sum(&args, t, 2, nullptr) == PP_OK);
    t[2].field.map = a;                                     // the map before it is b
    t[2].flags = PP_SUM_SAME_CELL;
    CHECK(pp_push_sum(&args, t, 3, nullptr) == PP_ERR_INVALID);
    for (pp_map* m : {a, twin, b}) CHECK(pp_map_destroy(m) == PP_OK);
}

// A map refused for its flags leaves nothing behind.
static void refused() {
    const std::vector<double> g = axis(5);
    std::vector<double> v(125 * 3);
    const double* parts[3] = {v.data(), v.data() + 125, v.data() + 250};
    pp_map* m = nullptr;
    CHECK(pp_map_create_parts(parts, 0, 3, 5, 5, 5, g.data(), g.data(), g.data(), 0.0, PP_MAP_NO_FP64 | PP_MAP_NO_FP32,
                              &m) == PP_ERR_INVALID);
    CHECK(m == nullptr && pp_release_staging() == PP_OK && used == 0);
}

int main(int argc, char** argv) {
    CHECK(argc == 2 && pp_init(0) == PP_OK);
    const std::string w = argv[1];
    if (w == "pieces") pieces();
    else if (w == "same_cell") same_cell();
    else if (w == "layout") layout();
    else if (w == "refused") refused();
    else CHECK(!"unknown case");
    return 0;
}
