// Which batches of tiny FP64 instances are solved by launches of whole
// iterations, and how long such a launch gets.
#include <cstdio>
#include <memory>
#include <string>
#include <vector>

#include "../../bnmf-algs_amd/csrc/bnmf_internal.hpp"
#include "fake_hip.hpp"

using namespace bnmf;

static int failures = 0;
#define CHECK(cond, ...)                       \
    do {                                       \
        if (!(cond)) {                         \
            ++failures;                        \
            std::printf("FAILED %s: ", #cond); \
            std::printf(__VA_ARGS__);          \
            std::printf("\n");                 \
        }                                      \
    } while (0)

struct Set {
    std::vector<double> X, ones;
    std::vector<InstSpec> specs;
    Set(uint32_t x, uint32_t y, uint32_t z, size_t n) : X((size_t)x * y, 2.0), ones(x + z, 1.0) {
        InstSpec s;
        s.x = x, s.y = y, s.z = z, s.X = X.data(), s.alpha = s.beta = ones.data();
        specs.assign(n, s);
    }
};

static std::vector<uint32_t> launches(uint32_t x, uint32_t y, uint32_t z, size_t n, size_t iters) {
    Set p(x, y, z, n);
    fake::reset();
    fake::tiny_iters.clear();
    Batch b(BNMF_F64, PSIM_F64_EXACT, 1e-50, p.specs);
    b.solve_async(iters);
    return fake::tiny_iters;
}

int main(int argc, char** argv) {
    fake::tiny = true;
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "route") {
        CHECK(!launches(8, 10, 3, 1, 10).empty(), "the fixture");
        CHECK(!launches(4, 32, 32, 256, 10).empty(), "some of few rows");
        CHECK(!launches(16, 32, 8, 2048, 10).empty(), "many of sixteen rows");
        CHECK(!launches(8, 8, 8, 2048, 10).empty(), "many small ones");
        CHECK(launches(4, 32, 32, 2048, 10).empty(), "many of few rows");
        CHECK(launches(4, 16, 64, 2048, 10).empty(), "many of few rows");
        CHECK(launches(70, 10, 3, 1, 10).empty(), "not of one tile");
    }
    if (failures) return 1;
    std::printf("tiny batches ok\n");
    return 0;
}
