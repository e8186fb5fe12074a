// Results to host memory (hostcopy.cpp): contents at every size class, pinned
// memory taken only by objects that fetch enough for it to pay, and once.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <thread>
#include <vector>

#include "../../bnmf-algs_amd/csrc/bnmf_internal.hpp"
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

static std::vector<char> pattern(size_t n) {
    std::vector<char> v(n);
    for (size_t i = 0; i < n; ++i) v[i] = (char)(i * 2654435761u >> 13);
    return v;
}

int main() {
    constexpr size_t MB = 1 << 20;
    const std::vector<char> src = pattern(70 * MB + 13);
    // one result: nothing is pinned below the size at which a pinned buffer
    // pays for itself at once
    for (size_t n : {(size_t)1, 4 * MB - 1, 8 * MB, 16 * MB + 5, 32 * MB}) {
        fake::reset();
        bnmf::HostStage st;
        std::vector<char> dst(n + 1, 77);
        st.copy(dst.data(), src.data(), n, nullptr);
        CHECK(fake::n_pins() == 0, "%zu bytes: %zu pinned", n, fake::n_pins());
        CHECK(std::memcmp(dst.data(), src.data(), n) == 0 && dst[n] == 77, "%zu bytes", n);
    }
    {  // a large one, twice
        fake::reset();
        bnmf::HostStage st;
        for (int rep = 0; rep < 2; ++rep) {
            std::vector<char> dst(src.size() + 1, 77);
            st.copy(dst.data(), src.data(), src.size(), nullptr);
            CHECK(std::memcmp(dst.data(), src.data(), src.size()) == 0 && dst[src.size()] == 77, "large");
        }
        CHECK(fake::n_pins() == 1, "%zu pinned", fake::n_pins());
    }
    {  // many results of ascending size from one object: pinned once
        fake::reset();
        bnmf::HostStage st;
        for (size_t n = MB; n < 40 * MB; n += 3 * MB + 17) {
            std::vector<char> dst(n);
            st.copy(dst.data(), src.data(), n, nullptr);
            CHECK(std::memcmp(dst.data(), src.data(), n) == 0, "%zu bytes", n);
        }
        CHECK(fake::n_pins() == 1, "%zu pinned", fake::n_pins());
    }
    {  // several threads
        bnmf::HostStage st;
        std::vector<std::thread> th;
        std::atomic<int> bad{0};
        for (int t = 0; t < 4; ++t)
            th.emplace_back([&, t] {
                for (size_t n : {3 * MB + t, 45 * MB + t, 9 * MB + t}) {
                    std::vector<char> dst(n);
                    st.copy(dst.data(), src.data() + t, n, nullptr);
                    if (std::memcmp(dst.data(), src.data() + t, n) != 0) ++bad;
                }
            });
        for (auto& t : th) t.join();
        CHECK(bad == 0, "%d", bad.load());
    }
    if (failures) return 1;
    std::printf("host copy ok\n");
    return 0;
}
