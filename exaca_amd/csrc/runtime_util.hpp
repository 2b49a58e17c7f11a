// runtime_util.hpp -- error plumbing shared by the C-ABI translation units: HIP status checks
// that throw, and the wrapper that turns exceptions into status codes at the boundary.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <stdexcept>
#include <string>

#include "../../include/exaca_ca.h"
#include "ca_common.hpp"

namespace exaca {

extern thread_local std::string g_last_error;

struct DeviceError : std::runtime_error {
    using std::runtime_error::runtime_error;
};
struct StateError : std::runtime_error {
    using std::runtime_error::runtime_error;
};

inline void hip_check(hipError_t e, const char *what) {
    if (e != hipSuccess) throw DeviceError(std::string(what) + ": " + hipGetErrorString(e));
}

// Device error flags (StepCtl::error) and their meaning, for the messages of the ABI calls.
inline std::string device_error_text(int flags) {
    std::string s = "device error flag " + std::to_string(flags) + " (";
    const char *sep = "";
    if (flags & 2) s += sep, s += "2: an active cell with GrainID 0", sep = ", ";
    if (flags & 16) s += sep, s += "16: a barrier wait that did not end within its bound", sep = ", ";
    if (flags & ~18) s += sep, s += "unknown bits";
    return s + ")";
}

// Workgroups of the frontier kernels of a plain-path handle: EXACA_BLOCKS (8 .. 2048, a multiple
// of 8) overrides the size-based choice, with two launches a step whatever the size. Tests narrow it
// so that a workgroup holds many claimants and the kernels' multi-round paths run.
inline int frontier_blocks_override() {
    const char *env = std::getenv("EXACA_BLOCKS");
    if (!env) return 0;
    const long v = std::strtol(env, nullptr, 10);
    if (v < 8 || v > 2048 || v % 8)
        throw std::invalid_argument("EXACA_BLOCKS must be a multiple of 8 in 8 .. 2048");
    return static_cast<int>(v);
}

// Claimants of a step that a team's workgroup stages in LDS: kTeamClaims, or fewer when EXACA_CAND_STAGE
// (1 .. 2048, read when a handle or an ensemble's slot is created) asks for it, so that tests can drive the
// path of those that do not fit on small domains.
inline uint32_t claim_stage() {
    const char *env = std::getenv("EXACA_CAND_STAGE");
    if (!env) return kTeamClaims;
    const long v = std::strtol(env, nullptr, 10);
    if (v < 1 || v > 2048) throw std::invalid_argument("EXACA_CAND_STAGE must be 1 .. 2048");
    return std::min(static_cast<uint32_t>(v), kTeamClaims);
}
// How long a team's workgroups wait for one another, in ticks of the 100 MHz clock: at the start of a launch
// (meet.hpp; EXACA_MEET_US) and at a barrier, at most (EXACA_BARRIER_US). The variables, 0 .. 40000000 us, are
// read when a handle or ensemble is created. Tests set 0: every launch is then left to one workgroup; the
// first barrier ends the domain with error 16.
inline uint32_t wait_ticks(const char *name, long us) {
    if (const char *env = std::getenv(name)) {
        char *end = nullptr;
        us = std::strtol(env, &end, 10);
        if (end == env || *end || us < 0 || us > 40000000)
            throw std::invalid_argument(std::string(name) + " must be 0 .. 40000000");
    }
    return static_cast<uint32_t>(us) * 100u;
}
inline uint32_t meet_wait_ticks() { return wait_ticks("EXACA_MEET_US", kMeetWait); }
inline uint32_t barrier_wait_ticks() { return wait_ticks("EXACA_BARRIER_US", kBarrierWait); }

template <typename F>
int guarded(F &&f) {
    try {
        f();
        return EXACA_OK;
    }
    catch (const DeviceError &e) {
        g_last_error = e.what();
        return EXACA_ERR_DEVICE;
    }
    catch (const StateError &e) {
        g_last_error = e.what();
        return EXACA_ERR_STATE;
    }
    catch (const std::exception &e) {
        g_last_error = e.what();
        return EXACA_ERR_INPUT;
    }
    catch (...) {
        g_last_error = "unknown error";
        return EXACA_ERR_INPUT;
    }
}

}  // namespace exaca

#define HIP_OK(x) ::exaca::hip_check((x), #x)
