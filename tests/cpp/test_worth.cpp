// LivePlan::worth, the host's look at a sample of X: a few busy columns or rows
// do not stand for a matrix that is otherwise empty, nor empty ones for a full
// matrix, whatever the width.
#include <cstdio>
#include <vector>

#include "../../bnmf-algs_amd/csrc/bnmf_internal.hpp"

using bnmf::LivePlan;

int main() {
    int failures = 0;
    auto check = [&](bool want, const std::vector<float>& X, size_t x, size_t y, const char* what) {
        const std::vector<double> D(X.begin(), X.end());
        for (bool got : {LivePlan::worth(BNMF_F32, X.data(), x, y, 0.4), LivePlan::worth(BNMF_F64, D.data(), x, y, 0.4)})
            if (got != want) ++failures, std::printf("FAILED %zu x %zu %s\n", x, y, what);
    };
    for (size_t x : {1, 7, 64, 100, 1024, 2048})
        for (size_t y : {1, 2, 63, 64, 100, 513, 1000, 1024, 2048}) {
            std::vector<float> X(x * y, 0.0f);
            check(true, X, x, y, "empty");
            std::fill(X.begin(), X.end(), 1.0f);
            check(false, X, x, y, "full");
            if (y < 63) continue;
            // busy columns: each alone, then every 64th, every 512th
            for (size_t c : {(size_t)0, (size_t)1, y / 2, y - 1}) {
                std::fill(X.begin(), X.end(), 0.0f);
                for (size_t i = 0; i < x; ++i) X[i * y + c] = 1.0f;
                check(true, X, x, y, "one busy column");
                for (float& v : X) v = 1.0f - v;
                check(false, X, x, y, "one empty column");
            }
            for (size_t s : {64, 512}) {
                std::fill(X.begin(), X.end(), 0.0f);
                for (size_t i = 0; i < x; ++i)
                    for (size_t j = 0; j < y; j += s) X[i * y + j] = 1.0f;
                check(true, X, x, y, "busy columns");
            }
            if (x < 64) continue;
            for (size_t r : {(size_t)0, x / 2, x - 1}) {
                std::fill(X.begin(), X.end(), 0.0f);
                for (size_t j = 0; j < y; ++j) X[r * y + j] = 1.0f;
                check(true, X, x, y, "one busy row");
            }
        }
    if (failures) return 1;
    std::printf("worth ok\n");
    return 0;
}
