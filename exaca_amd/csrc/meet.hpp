// meet.hpp -- how the workgroups of a team agree to step a domain together, or leave it to one of
// them (host and device).
//
// A team's barriers end only if all its workgroups run at once. Nothing grants that: each XCD starts the
// workgroups of every queue as it finds room, and where other launches (another ensemble, another
// process) fill the compute units, two launches can each hold the room that the other's team lacks.
// So a team meets before it touches the domain. Every workgroup has a word, in which it reports for the
// launch, and waits, for a bounded time, until all have reported: then all of them run, and every later
// barrier ends. One that has waited too long refuses those that have not reported, by a compare-and-swap
// of their words; then workgroup 0 takes the domain through the launch alone, and the others leave (also
// those that start later): their room serves other teams, and one workgroup waits for nobody.
// A word is reported or refused once in a launch, so where one was refused nobody ever sees all reported, and
// where all are reported none can be refused any more: all follow the same outcome. The words hold the
// launch's number, which only grows, and nothing needs to be cleared between launches.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace exaca {

enum class Meet { kTogether, kAlone, kLeave };
struct Met {
    bool all, refused;  // every word reported; some word refused
};

__host__ __device__ inline uint64_t meet_reported(uint64_t launch) { return 2 * launch; }
__host__ __device__ inline uint64_t meet_refused(uint64_t launch) { return 2 * launch + 1; }

// W: report() raises this workgroup's word to meet_reported (a maximum: a refused one stays); look() reads all;
// expired() whether it has waited long enough; refuse() swaps each word that look() found not reported, if
// it still is as found, for meet_refused.
template <typename W>
__host__ __device__ inline Meet meet(W &w, uint32_t b) {
    w.report();
    for (;;) {
        const Met m = w.look();
        if (m.refused) return b == 0 ? Meet::kAlone : Meet::kLeave;
        if (m.all) return Meet::kTogether;
        if (w.expired()) w.refuse();
    }
}

}  // namespace exaca
