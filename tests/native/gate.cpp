// Random launches of many problems on several streams: at every launch, no set
// of launches that may be under way together (none ordered before another, by
// its problem or by a wait) weighs more than the room.  Also checks the two
// ends: what fits together waits for nothing, what fills an XCD waits for all.
#include <cstdio>
#include <cstdlib>
#include <random>
#include <set>
#include <vector>

#include "resident_gate.hpp"

using namespace chysx_amd;

struct Launch {
    int owner, weight;
    std::set<int> before;  // launches ordered before it (transitive)
    bool done = false;
};

// the heaviest set of unordered launches among `left`, all unordered with the chosen ones
int heaviest(const std::vector<Launch>& all, const std::vector<int>& left) {
    if (left.empty()) return 0;
    const int x = left.back();
    std::vector<int> without(left.begin(), left.end() - 1), with;
    for (int y : without)
        if (!all[size_t(x)].before.count(y) && !all[size_t(y)].before.count(x)) with.push_back(y);
    return std::max(heaviest(all, without), all[size_t(x)].weight + heaviest(all, with));
}

#define EXPECT(c) \
    if (!(c)) { std::printf("failed: %s (line %d)\n", #c, __LINE__); return 1; }

int main() {
    const int room = gate_room(256);
    EXPECT(room == 31 && gate_room(4) == 0);
    EXPECT(gate_weight(256, 256, true, 256) == room && gate_weight(2, 2, true, 256) == 1);
    EXPECT(gate_weight(64, 64, true, 256) == 8 && gate_weight(2000, 8, true, 256) == 7);
    EXPECT(gate_weight(396, 198, false, 256) == room && gate_weight(100, 1, false, 256) == 0);
    long looked = 0, waited = 0;
    for (unsigned seed = 0; seed < 300; ++seed) {
        std::mt19937 rng(seed);
        auto pick = [&](int lo, int hi) { return std::uniform_int_distribution<int>(lo, hi)(rng); };
        GateBook<int> book;
        const int owners = pick(2, 7);
        std::vector<int> last(size_t(owners), -1), recorded(size_t(owners), -1);
        std::vector<Launch> all;
        char tokens[8];
        for (int step = 0; step < 60; ++step) {
            // some launches end, each after those before it
            for (Launch& L : all)
                if (!L.done && pick(0, 9) == 0) {
                    bool free = true;
                    for (int b : L.before) free = free && all[size_t(b)].done;
                    L.done = free;
                }
            const int o = pick(0, owners - 1), w = pick(0, 3) == 0 ? room : pick(1, room);
            // an owner's event stands for its latest launch
            const auto waits = book.admit(tokens + o, o, w, room,
                                          [&](int owner) { return all[size_t(recorded[size_t(owner)])].done; });
            Launch L{o, w, {}, false};
            auto behind = [&](int x) {
                L.before.insert(x);
                L.before.insert(all[size_t(x)].before.begin(), all[size_t(x)].before.end());
            };
            if (last[size_t(o)] >= 0) behind(last[size_t(o)]);
            for (int owner : waits) {
                EXPECT(owner != o);
                behind(recorded[size_t(owner)]);
                ++waited;
            }
            last[size_t(o)] = recorded[size_t(o)] = int(all.size());
            all.push_back(L);
            std::vector<int> open;
            for (size_t k = 0; k < all.size(); ++k)
                if (!all[k].done) open.push_back(int(k));
            if (open.size() > 18) open.erase(open.begin(), open.end() - 18);
            EXPECT(heaviest(all, open) <= room);
            ++looked;
        }
        EXPECT(book.size() <= size_t(owners));
    }
    GateBook<int> book;
    int a, b, c, d;
    const auto running = [](int) { return false; };
    EXPECT(book.admit(&a, 1, 8, room, running).empty() && book.admit(&b, 2, 8, room, running).empty());
    EXPECT(book.admit(&c, 3, 8, room, running).empty() && book.admit(&a, 1, 8, room, running).empty());
    EXPECT(book.admit(&d, 4, 8, room, running).size() == 1);
    EXPECT(book.admit(&a, 1, room, room, running).size() >= 2);
    EXPECT(book.admit(&b, 2, 1, room, running).size() == 1);
    std::printf("ok %ld %ld\n", looked, waited);
    return 0;
}
