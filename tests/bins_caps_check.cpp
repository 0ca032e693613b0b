// Checks bin_capacities (ohpic_bins.hpp): every bin holds its own count with
// the slack, a bin below its surroundings by a fluctuation is sized for their
// mean, a gradient adds at most four standard deviations, and the layout never
// exceeds the elements it is given where the plain one fits.
#include <cstdio>
#include <cstdlib>
#include <random>

#include "../ohhelppic3d_amd/csrc/ohpic_bins.hpp"

using namespace ohpic;

#define CHECK(c)                                              \
    do {                                                      \
        if (!(c)) {                                           \
            std::printf("line %d: %s\n", __LINE__, #c);      \
            return 1;                                         \
        }                                                     \
    } while (0)

int main()
{
    std::mt19937 rng(7);
    const int shapes[][3] = {{1, 1, 1}, {2, 1, 3}, {3, 3, 3}, {12, 13, 16}, {1, 40, 2}};
    for (const auto &nt : shapes) {
        const size_t n = (size_t)nt[0] * nt[1] * nt[2];
        for (double mean : {0.0, 3.0, 512.0, 20000.0}) {
            std::poisson_distribution<int64_t> p(mean > 0 ? mean : 1e-9);
            std::vector<int64_t> c(n);
            int64_t total = 0, plain = 0;
            for (auto &v : c) total += v = p(rng);
            for (int64_t v : c) plain += bin_capacity(v, 0.15);
            const auto e = expected_counts(c, nt);
            const auto cap = bin_capacities(c, nt, 0.15, (int64_t)1 << 40);
            const auto tight = bin_capacities(c, nt, 0.15, plain);
            int64_t sum = 0;
            for (size_t t = 0; t < n; ++t) {
                CHECK(e[t] >= c[t]);
                CHECK(e[t] <= c[t] + 4 * (int64_t)std::sqrt((double)c[t]) + 4);
                CHECK(cap[t] == bin_capacity(e[t], 0.15) && cap[t] % 64 == 0);
                sum += tight[t];
            }
            CHECK(sum <= plain);
            // bins that fluctuate around one mean: none far below it
            if (mean >= 512 && n > 27)
                for (size_t t = 0; t < n; ++t) CHECK((double)e[t] > mean - 1.5 * std::sqrt(mean));
        }
    }
    // a step in the density: the low side's bins keep to their own counts
    const int nt[3] = {8, 1, 1};
    std::vector<int64_t> c = {100, 100, 100, 100, 90000, 90000, 90000, 90000};
    const auto e = expected_counts(c, nt);
    CHECK(e[1] == 100 && e[3] == 144 && e[0] == 144 && e[5] == 90000);
    std::printf("ok\n");
    return 0;
}
