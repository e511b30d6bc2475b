// A model of how the workgroups of a one-launch batch solve come to run: each
// of 8 XCDs is given every 8th workgroup, in order, and starts the next one
// when one of its compute units is free; a cloth's workgroups keep theirs
// until all of them have started and the cloth is solved.  Prints, for each
// batch, how many of the random orders of events end with every workgroup
// waiting: with the placing that resident_by_start() picks, and in the order of
// starting.
#include <cstdio>
#include <deque>
#include <functional>
#include <random>
#include <vector>

#include "pcg_resident.hpp"

using namespace chysx_amd;

constexpr int kCus = 256;

bool stuck(const std::vector<int>& clusters, bool by_start, unsigned seed) {
    std::mt19937 rng(seed);
    std::vector<int> cloth;  // of a place
    for (size_t k = 0; k < clusters.size(); ++k) cloth.insert(cloth.end(), size_t(clusters[k]), int(k));
    const int n = int(cloth.size());
    std::vector<int> next(kXcds), left(kXcds, kCus / kXcds), started(clusters.size(), 0);
    std::vector<std::vector<int>> on(clusters.size(), std::vector<int>(kXcds, 0));
    std::vector<double> speed(kXcds);
    for (int x = 0; x < kXcds; ++x) {
        next[size_t(x)] = x;
        speed[size_t(x)] = std::uniform_real_distribution<double>(0.05, 1.0)(rng);
    }
    std::vector<int> running;
    int places = 0, done = 0;
    for (;;) {
        std::vector<double> weight(kXcds, 0.0);
        bool any = false;
        for (int x = 0; x < kXcds; ++x)
            if (next[size_t(x)] < n && left[size_t(x)] > 0) {
                weight[size_t(x)] = speed[size_t(x)];
                any = true;
            }
        // a solve lasts far longer than a start, but may end between two starts
        const bool finish = !running.empty() && (!any || std::uniform_int_distribution<int>(0, 99)(rng) == 0);
        if (finish) {
            const size_t q = std::uniform_int_distribution<size_t>(0, running.size() - 1)(rng);
            const int k = running[q];
            running.erase(running.begin() + long(q));
            for (int x = 0; x < kXcds; ++x) left[size_t(x)] += on[size_t(k)][size_t(x)];
            done += clusters[size_t(k)];
        } else if (any) {
            const int x = std::discrete_distribution<int>(weight.begin(), weight.end())(rng);
            const int id = next[size_t(x)], k = cloth[size_t(by_start ? places : id)];
            ++places;
            next[size_t(x)] += kXcds;
            --left[size_t(x)];
            ++on[size_t(k)][size_t(x)];
            if (++started[size_t(k)] == clusters[size_t(k)]) running.push_back(k);
        } else {
            return done < n;
        }
    }
}

void batch(const char* name, std::vector<int> clusters) {
    std::sort(clusters.begin(), clusters.end(), std::greater<int>());
    int wgs = 0;
    for (int c : clusters) wgs += c;
    const bool pick = resident_by_start(wgs, clusters[0], kCus);
    int as_picked = 0, by_start = 0;
    for (unsigned seed = 0; seed < 200; ++seed) {
        as_picked += stuck(clusters, pick, seed);
        by_start += stuck(clusters, true, seed);
    }
    std::printf("%s %d %d %d\n", name, pick ? 1 : 0, as_picked, by_start);
}

int main() {
    std::mt19937 rng(7);
    auto uneven = [&](int count, int lo, int hi) {
        std::vector<int> c;
        for (int k = 0; k < count; ++k) c.push_back(std::uniform_int_distribution<int>(lo, hi)(rng));
        return c;
    };
    batch("one256", {256});
    batch("two128", {128, 128});
    batch("two198", {198, 198});
    batch("two130", {130, 130});
    batch("three256", {256, 256, 256});
    batch("sixteen130", std::vector<int>(16, 130));
    batch("forty32", std::vector<int>(40, 32));
    batch("forty33", std::vector<int>(40, 33));
    batch("uneven16", uneven(300, 1, 16));
    batch("uneven32", uneven(200, 1, 32));
    batch("uneven256", uneven(60, 1, 256));
    return 0;
}
