// Packing the nonempty fibers takes as long as some dozens of iterations save:
// a plain call of fewer does not pack, one of many does, and so does a batch,
// which may be solved again.
#include <cstdio>
#include <vector>

#include "../../include/bnmf_hip.h"
#include "fake_hip.hpp"

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

int main() {
    struct Case {
        size_t x, y, z, few, many;
    };
    for (const Case& c : {Case{64, 64, 8, 8, 64}, Case{300, 300, 16, 8, 64}, Case{512, 512, 32, 16, 128},
                          Case{1024, 1024, 32, 32, 128}}) {
        std::vector<float> X(c.x * c.y, 0.0f), S(c.x * c.y * c.z);
        for (size_t t = 0; t < X.size(); t += 11) X[t] = 2.0f;
        std::vector<double> alpha(c.x, 1.0), beta(c.z, 1.0);
        auto packs = [&](size_t iters) {
            fake::reset();
            const bnmf_status st = bnmf_bld_mult_f32(X.data(), c.x, c.y, c.z, alpha.data(), beta.data(), iters, 1, 1e-50,
                                                     nullptr, 1, S.data());
            CHECK(st == BNMF_OK, "%d", (int)st);
            return fake::packs.load();
        };
        for (size_t it : {(size_t)0, (size_t)1, c.few}) CHECK(packs(it) == 0, "%zu x %zu x %zu, %zu iterations", c.x, c.y, c.z, it);
        CHECK(packs(c.many) == 1, "%zu x %zu x %zu, %zu iterations", c.x, c.y, c.z, c.many);
        fake::reset();
        bnmf_bld_desc d{};
        d.x = c.x, d.y = c.y, d.z = c.z, d.X = X.data(), d.alpha = alpha.data(), d.beta = beta.data(), d.a = d.b = 1.0;
        bnmf_batch* b = nullptr;
        CHECK(bnmf_batch_create(&b, BNMF_F32, &d, 1, 1, 1e-50) == BNMF_OK, "batch");
        CHECK(fake::packs == 1, "batch");
        bnmf_batch_destroy(b);
    }
    if (failures) return 1;
    std::printf("few iterations ok\n");
    return 0;
}
