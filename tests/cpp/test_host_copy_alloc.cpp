// Results to host memory (hostcopy.cpp) where host memory runs out: the copy is
// complete or throws, and the process goes on.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <vector>

#include "../../bnmf-algs_amd/csrc/bnmf_internal.hpp"
#include "fake_hip.hpp"

static std::atomic<long> g_fail_new{-1};  // allocations left until one fails
void* operator new(size_t n) {
    if (g_fail_new.load() >= 0 && g_fail_new.fetch_sub(1) == 0) throw std::bad_alloc();
    void* p = std::malloc(n);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

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

static std::vector<char> pattern(size_t n) {
    std::vector<char> v(n);
    for (size_t i = 0; i < n; ++i) v[i] = (char)(i * 2654435761u >> 13);
    return v;
}

int main() {
    constexpr size_t MB = 1 << 20;
    const std::vector<char> src = pattern(48 * MB);
    for (long k = 0; k < 40; ++k) {
        bnmf::HostStage st;
        std::vector<char> dst(48 * MB);
        st.copy(dst.data(), src.data(), dst.size(), nullptr);
        std::fill(dst.begin(), dst.end(), 0);
        bool done = false;
        g_fail_new = k;
        try {
            st.copy(dst.data(), src.data(), dst.size(), nullptr);
            done = true;
        } catch (const std::bad_alloc&) {
        }
        g_fail_new = -1;
        CHECK(!done || std::memcmp(dst.data(), src.data(), dst.size()) == 0, "after allocation %ld", k);
    }
    if (failures) return 1;
    std::printf("host copy alloc ok\n");
    return 0;
}
