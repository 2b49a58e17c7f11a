// meet.hpp -- how the workgroups of a team agree to step a domain together, or leave it to one of
// them (host and device).
//
// A team's barriers end only if all its workgroups run at once. Nothing grants that: each XCD starts the
// workgroups of every queue as it finds room, and where other launches (another ensemble, another
// process) fill the compute units, two launches can each hold the room that the other's team lacks.
// So a team meets before it touches the domain. Every workgroup reports and waits, for a bounded time,
// until all have: then all of them run, and every later barrier ends. The first that has waited too long
// settles instead that workgroup 0 takes the domain through the launch alone, and the others leave
// (also those that start later): their room serves other teams, and one workgroup waits for nobody.
// One compare-and-swap of the decision word settles it, so all follow the same decision. A decision and a
// report carry the number of the launch, and nothing needs to be cleared between launches.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace exaca {

enum class Meet { kTogether, kAlone, kLeave };

__host__ __device__ inline uint64_t meet_decision(uint32_t launch, bool together) {
    return static_cast<uint64_t>(launch) << 1 | (together ? 1u : 0u);
}
// W: report() posts this workgroup's; decision() and all_reported() read; expired() whether it has waited
// long enough; settle(from, to) stores the decision `to` if it is still `from` and gives the one found.
template <typename W>
__host__ __device__ inline Meet meet(const W &w, uint32_t b, uint32_t launch) {
    w.report();
    uint64_t d = w.decision();
    while (d >> 1 != launch) {
        const bool all = w.all_reported();
        if (all || w.expired()) {
            const uint64_t mine = meet_decision(launch, all), found = w.settle(d, mine);
            d = found == d ? mine : found;  // the first one stands
        }
        else
            d = w.decision();
    }
    return d & 1u ? Meet::kTogether : (b == 0 ? Meet::kAlone : Meet::kLeave);
}

}  // namespace exaca
