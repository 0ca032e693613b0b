// Checks ohpic_plan.hpp: load_level against its definition, the tiles' order
// against a comparison sort by level, the chunk limits of a plan, and that a
// plan takes well below the time of a comparison sort that takes the levels as
// it compares.
#include <chrono>
#include <cmath>
#include <cstdio>
#include <random>

#include "../ohhelppic3d_amd/csrc/ohpic_plan.hpp"

using namespace ohpic;

#define CHECK(c)                                        \
    do {                                                \
        if (!(c)) {                                     \
            std::printf("line %d: %s\n", __LINE__, #c); \
            return 1;                                   \
        }                                               \
    } while (0)

static int level(int64_t l) { return l <= 0 ? -1 : (int)std::floor(8.0 * std::log2((double)l)); }

static void by_comparison(std::vector<TileLoad> &t)
{
    std::stable_sort(t.begin(), t.end(), [](const TileLoad &a, const TileLoad &b) {
        return level(a.load) > level(b.load);
    });
}

template <class F>
static double best_us(const std::vector<TileLoad> &tiles, F f)
{
    double best = 1e30;
    for (int r = 0; r < 15; ++r) {
        std::vector<TileLoad> t(tiles);
        const auto t0 = std::chrono::steady_clock::now();
        f(t);
        best = std::min(best, std::chrono::duration<double, std::micro>(
                                  std::chrono::steady_clock::now() - t0).count());
    }
    return best;
}

int main()
{
    std::mt19937_64 rng(3);
    for (int64_t l = -3; l < 200000; ++l) CHECK(load_level(l) == level(l));
    for (int k = 0; k < 200000; ++k) {
        const int64_t l = (int64_t)(rng() >> (64 - 40)) >> (rng() % 30);
        CHECK(load_level(l) == level(l));
    }
    CHECK(load_level(INT64_MAX) == 8 * 62 + 7);
    for (int k = 0; k < 62; ++k) CHECK(load_level((int64_t)1 << k) == 8 * k);

    for (int n : {0, 1, 2, 63, 2496, 32768}) {
        for (double spread : {0.0, 0.05, 1.0}) {
            std::lognormal_distribution<double> d(std::log(2000.0), spread);
            std::vector<TileLoad> tiles;
            for (int i = 0; i < n; ++i)
                tiles.push_back({i % 3, i, rng() % 50 == 0 ? 0 : (int64_t)d(rng) / 64 * 64});
            std::vector<TileLoad> a(tiles), b(tiles);
            std::vector<int> nch;
            by_comparison(b);
            for (int64_t slots : {1, 768, 100000}) {
                a = tiles;
                plan_chunks(a, slots, 2048, nch);
                CHECK(a.size() == b.size() && nch.size() == a.size());
                int64_t extra = 0;
                for (int i = 0; i < n; ++i) {
                    CHECK(a[i].inst == b[i].inst && a[i].tile == b[i].tile && a[i].load == b[i].load);
                    CHECK(nch[i] >= 1 && nch[i] <= 256);
                    CHECK(nch[i] == 1 || a[i].load / nch[i] >= kMinChunkLoad);
                    extra += nch[i] - 1;
                }
                CHECK(extra <= 2048);
            }
            if (n < 2000) continue;
            const double plan = best_us(tiles, [&](std::vector<TileLoad> &t) { plan_chunks(t, 768, 0, nch); });
            const double sort = best_us(tiles, by_comparison);
            std::printf("%d tiles, spread %.2f: plan %.0f us, comparison sort %.0f us\n", n, spread,
                        plan, sort);
            if (spread > 0.5) CHECK(plan < 0.5 * sort);
        }
    }
    std::printf("ok\n");
    return 0;
}
