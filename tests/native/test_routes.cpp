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

int main(int argc, char** argv) {
    CHECK(argc == 2);
    const std::string w = argv[1];
    if (w == "gather") gather();
    else CHECK(!"unknown case");
    return 0;
}
