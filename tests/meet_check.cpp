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
    std::atomic<uint64_t> word[64];
};
struct Group {
    Words &words;
    uint32_t b, nb;
    uint64_t launch;
    int looks;  // until the wait expires (negative: never)
    uint64_t seen[64] = {};
    void report() {
        uint64_t v = words.word[b].load();
        while (v < exaca::meet_reported(launch) &&
               !words.word[b].compare_exchange_weak(v, exaca::meet_reported(launch), std::memory_order_relaxed)) {
        }
    }
    exaca::Met look() {
        std::this_thread::yield();
        exaca::Met m{true, false};
        for (uint32_t i = 0; i < nb; i++) {
            seen[i] = words.word[i].load(std::memory_order_relaxed);
            m.all = m.all && seen[i] == exaca::meet_reported(launch);
            m.refused = m.refused || seen[i] == exaca::meet_refused(launch);
        }
        return m;
    }
    bool expired() { return looks >= 0 && (looks == 0 || looks-- == 0); }
    void refuse() {
        for (uint32_t i = 0; i < nb; i++)
            if (seen[i] < exaca::meet_reported(launch)) {
                uint64_t was = seen[i];
                words.word[i].compare_exchange_strong(was, exaca::meet_refused(launch), std::memory_order_relaxed);
            }
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
                        Group g{words, b, nb, static_cast<uint64_t>(launch), looks[b]};
                        role[b] = exaca::meet(g, b);
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
