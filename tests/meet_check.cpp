// Checks the meeting of a team's workgroups (meet.hpp) with a thread per workgroup: team sizes 2 .. 64, many
// launches on the same words, waits that expire after a random number of looks (some at once, some never),
// and workgroups that start only when others of the team have left, as they do when those hold the room
// they need. In every launch either all take the domain together, or workgroup 0 alone and all others leave;
// and where nobody's wait expires, all take it. Prints the launches of each kind and exits nonzero on any
// other outcome.
#include <algorithm>
#include <atomic>
#include <cstdio>
#include <random>
#include <thread>
#include <vector>

#include "meet.hpp"

using exaca::Meet;

struct Words {
    std::atomic<uint32_t> report[64];
    std::atomic<uint64_t> decision;
};
struct Group {
    Words &words;
    uint32_t b, nb, launch;
    mutable int looks;  // until the wait expires (negative: never)
    void report() const { words.report[b].store(launch, std::memory_order_relaxed); }
    uint64_t decision() const {
        std::this_thread::yield();
        return words.decision.load(std::memory_order_relaxed);
    }
    bool all_reported() const {
        for (uint32_t i = 0; i < nb; i++)
            if (words.report[i].load(std::memory_order_relaxed) != launch) return false;
        return true;
    }
    bool expired() const { return looks >= 0 && looks-- == 0; }
    uint64_t settle(uint64_t from, uint64_t to) const {
        words.decision.compare_exchange_strong(from, to, std::memory_order_relaxed);
        return from;
    }
};

int main() {
    std::mt19937 rng(5);
    int together = 0, alone = 0, wrong = 0;
    for (uint32_t nb : {2u, 3u, 8u, 16u, 64u}) {
        Words words{};
        const int launches = 12000 / static_cast<int>(nb);
        for (int launch = 1; launch <= launches; launch++) {
            const int kind = launch % 4;  // 0: nobody's wait expires; 1: short waits; 2: at once; 3: late starters
            std::vector<Meet> role(nb, Meet::kLeave);
            std::vector<int> looks(nb);
            std::vector<uint32_t> order(nb);
            for (uint32_t b = 0; b < nb; b++) {
                looks[b] = kind == 0 ? -1 : (kind == 2 ? 0 : static_cast<int>(rng() % 40));
                order[b] = b;
            }
            std::shuffle(order.begin(), order.end(), rng);
            const uint32_t first = kind == 3 ? 1 + rng() % nb : nb;
            for (uint32_t part : {0u, first}) {  // the rest start when the first ones have left
                std::vector<std::thread> run;
                for (uint32_t i = part; i < (part ? nb : first); i++)
                    run.emplace_back([&, b = order[i]] {
                        const Group g{words, b, nb, static_cast<uint32_t>(launch), looks[b]};
                        role[b] = exaca::meet(g, b, static_cast<uint32_t>(launch));
                    });
                for (std::thread &t : run) t.join();
                if (first == nb) break;
            }
            uint32_t n = 0;
            for (Meet m : role) n += m == Meet::kTogether;
            bool by_one = role[0] == Meet::kAlone;
            for (uint32_t b = 1; b < nb; b++) by_one = by_one && role[b] == Meet::kLeave;
            if (n == nb) together++;
            else if (by_one && kind != 0) alone++;
            else wrong++;
            if (kind == 3 && first < nb && n) wrong++;
        }
    }
    std::printf("together %d alone %d wrong %d\n", together, alone, wrong);
    return wrong || !together || !alone;
}
