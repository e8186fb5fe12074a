// Batches at the limit of device memory: what is taken only for speed (packed
// fibers, lists of nonempty entries, the partial sums of short tiles) never
// makes a batch fail that would fit without it.
#include <cstdio>
#include <functional>
#include <memory>
#include <random>
#include <vector>

#include "../../bnmf-algs_amd/csrc/bnmf_internal.hpp"
#include "fake_hip.hpp"

using namespace bnmf;

static int failures = 0;
#define CHECK(cond, ...)                          \
    do {                                          \
        if (!(cond)) {                            \
            ++failures;                           \
            std::printf("FAILED %s: ", #cond);    \
            std::printf(__VA_ARGS__);             \
            std::printf("\n");                    \
        }                                         \
    } while (0)

template <typename T>
struct Problem {
    std::vector<T> X;
    std::vector<double> alpha, beta;
    uint32_t x, y, z;
    Problem(uint32_t x_, uint32_t y_, uint32_t z_, double share, unsigned seed) : alpha(x_, 1.0), beta(z_, 1.0), x(x_), y(y_), z(z_) {
        std::mt19937 g(seed);
        std::uniform_real_distribution<double> u(0, 1);
        X.resize((size_t)x * y);
        for (T& v : X) v = u(g) < share ? T(3) : T(0);
    }
};

// the smallest capacity at which make() succeeds
static size_t least_capacity(const std::function<void()>& make, size_t hi) {
    size_t lo = 0;
    while (hi - lo > 256) {
        const size_t mid = lo + (hi - lo) / 2;
        fake::reset(mid);
        try {
            make();
            hi = mid;
        } catch (const Error&) {
            lo = mid;
        }
    }
    return hi;
}

// lean: the same batch where nothing extra is wanted
static void check(const char* what, const std::function<void()>& make, const std::function<void()>& lean) {
    fake::reset();
    make();
    CHECK(fake::in_use() == 0, "%s: %zu bytes left", what, fake::in_use());
    const size_t n = fake::n_mallocs();
    for (size_t k = 1; k <= n; ++k) {
        fake::reset(~(size_t)0, k);
        try {
            make();
        } catch (const Error& e) {
            CHECK(false, "%s: allocation %zu of %zu failing once: %s", what, k, n, e.what());
        }
        CHECK(fake::in_use() == 0, "%s: %zu bytes left after allocation %zu failed", what, fake::in_use(), k);
    }
    const size_t most = (size_t)1 << 30, floor = least_capacity(lean, most);
    for (size_t cap = floor; cap < 3 * floor; cap += floor / 60) {
        fake::reset(cap);
        try {
            make();
        } catch (const Error& e) {
            CHECK(false, "%s: fails in %zu bytes, fits in %zu without extras: %s", what, cap, floor, e.what());
            break;
        }
    }
    fake::reset();
}

template <typename T>
static void batches(int dtype) {
    std::vector<Problem<T>> p;
    p.emplace_back(100, 150, 16, 0.05, 1);
    p.emplace_back(90, 60, 40, 0.1, 2);
    p.emplace_back(64, 64, 8, 0.9, 3);
    auto make = [&](double eps) {
        std::vector<InstSpec> s;
        for (auto& q : p) {
            InstSpec i;
            i.x = q.x, i.y = q.y, i.z = q.z, i.X = q.X.data(), i.alpha = q.alpha.data(), i.beta = q.beta.data();
            s.push_back(i);
        }
        Batch b(dtype, dtype == BNMF_F32 ? PSIM_F32 : PSIM_F64_EXACT, eps, s);
        b.solve_async(40);
        b.synchronize();
    };
    // eps below 1e-200 is not for the packed form
    check(dtype == BNMF_F32 ? "Batch FP32" : "Batch FP64", [&] { make(1e-50); }, [&] { make(1e-250); });
}

static void appr() {
    std::vector<Problem<double>> p;
    p.emplace_back(100, 150, 16, 0.05, 1);
    p.emplace_back(90, 60, 40, 0.9, 2);
    auto make = [&](double eps) {
        std::vector<ApprSpec> s;
        for (auto& q : p) {
            ApprSpec i;
            i.x = q.x, i.y = q.y, i.z = q.z, i.X = q.X.data(), i.alpha = q.alpha.data(), i.beta = q.beta.data();
            s.push_back(i);
        }
        ApprBatch b(BNMF_F64, eps, s);
        b.solve_async(5);
        b.synchronize();
    };
    check("ApprBatch FP64", [&] { make(1e-50); }, [&] { make(1e-250); });
}

int main() {
    batches<float>(BNMF_F32);
    batches<double>(BNMF_F64);
    appr();
    if (failures) return 1;
    std::printf("batch memory ok\n");
    return 0;
}
