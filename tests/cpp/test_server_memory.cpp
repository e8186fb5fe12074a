// The solve server's optional memory: packed fibers never fail a request, never
// keep a later one waiting that fits beside the dense tensors, and cost no
// allocation, copy or launch per request and step.
#include <cstdio>
#include <cstring>
#include <random>
#include <string>
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

struct Problem {
    std::vector<float> X, S;
    std::vector<double> alpha, beta;
    bnmf_bld_desc d{};
    Problem(size_t x, size_t y, size_t z, double share) : X(x * y), S(x * y * z), alpha(x, 1.0), beta(z, 1.0) {
        std::mt19937 g(x + y);
        std::uniform_real_distribution<double> u(0, 1);
        for (float& v : X) v = u(g) < share ? 2.0f : 0.0f;
        d.x = x, d.y = y, d.z = z, d.X = X.data(), d.alpha = alpha.data(), d.beta = beta.data(), d.a = d.b = 1.0;
    }
    size_t bytes() const { return bnmf_server_request_bytes(BNMF_F32, d.x, d.y, d.z); }
};

static uint64_t submit(bnmf_server* s, Problem& p, size_t iters) {
    uint64_t t = 0;
    CHECK(bnmf_server_submit(s, &p.d, iters, 0, &t) == BNMF_OK, "submit");
    return t;
}

// no device memory left once the server is warm
static void full_device() {
    fake::reset();
    bnmf_server* s = nullptr;
    Problem dense(200, 150, 16, 1.0), sparse(200, 150, 16, 0.05);
    CHECK(bnmf_server_create(&s, BNMF_F32, 16 * dense.bytes(), 0, 1, 1e-50) == BNMF_OK, "create");
    const uint64_t t0 = submit(s, dense, 100);
    CHECK(bnmf_server_wait(s, t0, 30.0) == BNMF_OK, "dense");
    fake::reset(fake::in_use());
    const uint64_t t1 = submit(s, sparse, 100);
    CHECK(bnmf_server_wait(s, t1, 30.0) == BNMF_OK, "a packable request on a full device");
    const uint64_t t2 = submit(s, dense, 100);
    CHECK(bnmf_server_wait(s, t2, 30.0) == BNMF_OK, "the next one");
    // room for the packing's own scratch, not for longer work lists; several at once
    fake::reset(fake::in_use() + 16384);
    std::vector<uint64_t> t;
    for (int k = 0; k < 6; ++k) {
        t.push_back(submit(s, k % 3 ? sparse : dense, 30 + 10 * k));
        if (k == 2) CHECK(bnmf_server_wait(s, t[0], 30.0) == BNMF_OK, "the first of several");
    }
    for (uint64_t k : t) CHECK(bnmf_server_wait(s, k, 30.0) == BNMF_OK, "one of several");
    bnmf_server_destroy(s);
    fake::reset();
    CHECK(fake::in_use() == 0, "%zu bytes left", fake::in_use());
}

// a later request that fits beside the dense tensors starts at once
static void later_request() {
    Problem a(300, 250, 24, 0.08), b(220, 250, 24, 0.08);
    bnmf_server* s = nullptr;
    CHECK(bnmf_server_create(&s, BNMF_F32, a.bytes() + b.bytes(), 0, 1, 1e-50) == BNMF_OK, "create");
    const uint64_t ta = submit(s, a, (size_t)1 << 40);
    bnmf_server_stats st{};
    for (int k = 0; k < 10000000 && (st.steps < 3 || st.bytes_in_use <= a.bytes()); ++k) bnmf_server_get_stats(s, &st);
    CHECK(st.bytes_in_use > a.bytes(), "not packed: %zu of %zu bytes", (size_t)st.bytes_in_use, a.bytes());
    const uint64_t tb = submit(s, b, 200);
    CHECK(bnmf_server_wait(s, tb, 20.0) == BNMF_OK, "waits for the packed one");
    int done = 1;
    bnmf_server_poll(s, ta, &done);
    CHECK(done == 0, "the long one ended");
    bnmf_server_get_stats(s, &st);
    CHECK(st.peak_active == 2, "%zu", (size_t)st.peak_active);
    bnmf_server_destroy(s);
}

// many small requests
static void small_requests() {
    constexpr size_t n = 64, iters = 160;
    Problem p(64, 64, 8, 0.05);
    bnmf_server* s = nullptr;
    CHECK(bnmf_server_create(&s, BNMF_F32, 4 * n * p.bytes(), 0, 1, 1e-50) == BNMF_OK, "create");
    CHECK(bnmf_server_wait(s, submit(s, p, iters), 30.0) == BNMF_OK, "warm");
    fake::reset();
    bnmf_server_stats a{}, b{};
    bnmf_server_get_stats(s, &a);
    std::vector<uint64_t> t;
    for (size_t k = 0; k < n; ++k) t.push_back(submit(s, p, iters));
    for (uint64_t k : t) CHECK(bnmf_server_wait(s, k, 30.0) == BNMF_OK, "request");
    bnmf_server_get_stats(s, &b);
    const size_t steps = b.steps - a.steps;
    CHECK(fake::packs > 0, "nothing packed");
    CHECK(fake::n_mallocs() <= 16, "%zu allocations for %zu requests", fake::n_mallocs(), n);
    // inputs of a request, the packing of those admitted together, a step's lists
    CHECK(fake::copies <= 3 * n + 12 * steps, "%zu copies in %zu steps", fake::copies.load(), steps);
    bnmf_server_destroy(s);
}

// the scheduler keeps to its own streams: copies of results to callers run on the
// null stream, and it would wait for them there
static void own_streams() {
    Problem p(300, 250, 24, 0.08);
    bnmf_server* s = nullptr;
    CHECK(bnmf_server_create(&s, BNMF_F32, 4 * p.bytes(), 0, 1, 1e-50) == BNMF_OK, "create");
    fake::reset();
    CHECK(bnmf_server_wait(s, submit(s, p, 100), 30.0) == BNMF_OK, "request");
    CHECK(fake::packs > 0, "nothing packed");
    CHECK(fake::on_null == 0, "%zu operations on the null stream", fake::on_null.load());
    bnmf_server_destroy(s);
}

// requests of few iterations are not packed, others are
static void few_iterations() {
    bnmf_server* s = nullptr;
    CHECK(bnmf_server_create(&s, BNMF_F32, (size_t)1 << 28, 0, 1, 1e-50) == BNMF_OK, "create");
    Problem small(64, 64, 8, 0.05), large(512, 300, 32, 0.05);
    for (Problem* p : {&small, &large})
        for (size_t iters : {0, 1, 8, 64}) {
            fake::reset();
            CHECK(bnmf_server_wait(s, submit(s, *p, iters), 30.0) == BNMF_OK, "request");
            CHECK((fake::packs > 0) == (iters == 64), "%zu iterations: packed %zu", iters, fake::packs.load());
        }
    bnmf_server_destroy(s);
}

int main(int argc, char** argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "full") full_device();
    if (what == "later") later_request();
    if (what == "small") small_requests();
    if (what == "few") few_iterations();
    if (what == "streams") own_streams();
    if (failures) return 1;
    std::printf("server memory ok\n");
    return 0;
}
