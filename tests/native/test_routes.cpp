// Rules of the dispatch that need no device: see test_native_cpu.py for the cases.
#include <stdio.h>
#include <string>

#include "hip_on_host.h"

#include "pp_copy.hip"
#include "pp_host.hip"

// which launches gather per lane: the lines lie at whole wavefronts per SIMD of 256 CUs (65536 particles each)
static void gather() {
    const int64_t one = 65536;
    const struct {
        int precision;
        bool rk4;
        int64_t limit;
    } want[] = {{PP_PREC_FP32_MIXED, false, 2 * one}, {PP_PREC_FP32_MIXED, true, one},
                {PP_PREC_FP64_FAST, false, one}, {PP_PREC_FP64_FAST, true, 0}};
    for (const auto& w : want)
        for (int64_t n : {(int64_t)1, one - 1, one, one + 1, 2 * one, 2 * one + 1})
            CHECK(gather_direct(n, w.precision, w.rk4) == (n <= w.limit));
}

// node indexes of the lean lookup, up to the 2^32 - 1 nodes it admits (-ftrapv: signed overflow aborts)
__attribute__((noinline)) static uint32_t index_of(const volatile int* q) {
    return node_index32(q[0], q[1], q[2], q[3], q[4]);
}

static void node_index() {
    const struct {
        int q[5];
        uint32_t want;
    } cases[] = {{{0, 0, 0, 7, 9}, 0u}, {{1, 2, 3, 7, 9}, 84u}, {{0, 65536, 65534, 65537, 65535}, 4294967294u},
                 {{2, 46340, 30891, 46341, 30892}, 4294698515u}, {{1290, 1290, 1290, 1291, 1291}, 2151685170u}};
    for (const auto& c : cases) CHECK(index_of(c.q) == c.want);
}

// a looping kernel's grid: enough blocks for few items, fewer than 2^32 threads for any number
static void grids() {
    for (int64_t n : {(int64_t)0, (int64_t)1, (int64_t)256, (int64_t)257, (int64_t)1 << 24, ((int64_t)1 << 24) + 1,
                      (int64_t)720000000 * 6, (int64_t)6 << 31}) {
        const uint64_t threads = (uint64_t)loop_blocks(n) * 256;
        CHECK(threads >= 256 && threads < ((uint64_t)1 << 32));
        CHECK(threads >= (uint64_t)n || threads == ((uint64_t)1 << 24));
        CHECK(threads < (uint64_t)n + 256 || n == 0);
    }
}

int main(int argc, char** argv) {
    CHECK(argc == 2);
    const std::string w = argv[1];
    if (w == "gather") gather();
    else if (w == "node_index") node_index();
    else if (w == "grids") grids();
    else CHECK(!"unknown case");
    return 0;
}
