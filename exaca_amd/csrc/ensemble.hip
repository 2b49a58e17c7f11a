// ensemble.hip -- many CA domains resident on one GPU, stepped together.
//
// Each domain occupies one slot: its state lives in a sub-range of a single device arena, and its
// DomainView sits in a device-resident slot table. A launch runs many steps of every domain: a team of
// workgroups takes each domain through them on its own (k_steps_n), so no domain waits for another
// once its team has met (meet.hpp), and the larger a domain, the larger its team (share_out). Every domain keeps its
// own cycle, control block and calendar, and stops itself on the device at the first 1000-step check
// with no liquid left, so each one evolves exactly as it would alone on the plain path. The host
// admits new domains into free slots between launches (continuous batching) and polls the
// per-slot status words after each.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <map>
#include <memory>
#include <vector>

#include "../../include/exaca_ca.h"
#include "ca_common.hpp"
#include "ca_kernels.hpp"
#include "deck.hpp"
#include "growth.hpp"
#include "init.hpp"
#include "runtime_util.hpp"

namespace exaca {
void upload_cells(const DomainView &d, const HostDomain &hd, uint8_t *melted, hipStream_t s);
StepCtl initial_ctl(const HostDomain &hd);
void download_field(const DomainView &d, int field, void *dst, size_t dst_bytes, hipStream_t s);
void layer_sites(const HostDomain &hd, int layer, std::vector<int32_t> &loc, std::vector<int32_t> &time);
}  // namespace exaca

namespace {

using exaca::DeviceError;
using exaca::StateError;
using exaca::guarded;

constexpr int kChunk = 50;         // steps are rounded up to this (even: parity 0 at launch boundaries)
constexpr int kMaxLaunch = 1000;   // most steps of one launch (a multiple of kChunk)
constexpr int kMaxBlocks = 256;    // largest workgroups-per-slot setting (above kMaxTeam: as kMaxTeam)
constexpr size_t kAlign = 256;

size_t up(size_t n) { return (n + kAlign - 1) / kAlign * kAlign; }

// First-fit allocator over the arena's byte range.
struct Arena {
    char *base = nullptr;
    size_t bytes = 0;
    std::map<size_t, size_t> free;  // offset -> length
    bool take(size_t n, size_t &off) {
        for (auto it = free.begin(); it != free.end(); ++it)
            if (it->second >= n) {
                off = it->first;
                const size_t rest = it->second - n;
                free.erase(it);
                if (rest) free[off + n] = rest;
                return true;
            }
        return false;
    }
    void give(size_t off, size_t n) {
        auto it = free.emplace(off, n).first;
        auto nx = std::next(it);
        if (nx != free.end() && it->first + it->second == nx->first) {
            it->second += nx->second;
            free.erase(nx);
        }
        if (it != free.begin()) {
            auto pv = std::prev(it);
            if (pv->first + pv->second == it->first) {
                pv->second += it->second;
                free.erase(it);
            }
        }
    }
    size_t available() const {
        size_t s = 0;
        for (auto &kv : free) s += kv.second;
        return s;
    }
};

// Device bytes one domain needs (state, frontier lists, tables, control).
size_t domain_bytes(const exaca::HostDomain &h, size_t ngrow, size_t nsums) {
    const size_t n = static_cast<size_t>(h.ncell);
    exaca::DomainView v{};
    exaca::set_geometry(v, h.X, h.Y, h.nz, h.nzA);
    size_t b = 0;
    b += up(sizeof(exaca::Cell) * n) + up(sizeof(exaca::Octa) * n);  // cell records
    b += 2 * up(4 * exaca::claim_entries(v, exaca::kMaxTeam)) + up(4 * exaca::kSyncWords);  // claim lists, team words
    b += 2 * up(4 * std::max<size_t>(h.nloc.size(), 1)) + up(8 * ngrow) + up(4 * nsums);
    b += up(sizeof(exaca::StepCtl)) + up(sizeof(exaca::StepStats)) + up(8ull * exaca::kPartRows * exaca::kMaxTeam);
    b += up(4 * exaca::kAlarmSlots * exaca::alarm_stride(h.ncell));  // calendar
    return b;
}

}  // namespace

// A domain initialised on the host, ready to be admitted.
struct exaca_prepared {
    exaca::Deck deck;
    exaca::HostDomain host;
    std::vector<double> grow;
    int ksat = 0;
    exaca::GrowthSums sums;
    long long liquid0 = 0;
    size_t bytes = 0;
};

struct exaca_ensemble {
    hipStream_t stream = nullptr;
    int slots = 0;
    int blocks = 64;      // workgroups per slot, at most
    int cus = 0;          // compute units, each of which holds one workgroup of a team
    Arena arena;
    exaca::DomainView *views_d = nullptr;
    std::vector<exaca::DomainView> views;
    int32_t *status_d = nullptr;  // per slot: final cycle (slots words), then error flags (slots words)
    std::vector<int32_t> status;  // both, as last polled
    std::vector<size_t> off, len;
    std::vector<char> used;
    std::vector<exaca::StepStats *> stats_d;
    // tables shared by every slot (one orientation file per ensemble)
    std::string orientation_file;
    float *guv = nullptr, *seed_cdl = nullptr;
    // The workgroups of a launch, for the domains that run now (dirty: to be shared out afresh)
    exaca::TeamPlace *places_d = nullptr;
    std::vector<exaca::TeamPlace> places;
    size_t places_cap = 0;
    bool dirty = true;
    long long steps = 0;
    uint64_t launches = 0;
    uint32_t meet_wait = 0, barrier_wait = 0;  // ticks

    ~exaca_ensemble() {
        if (arena.base) (void)hipFree(arena.base);
        if (views_d) (void)hipFree(views_d);
        if (places_d) (void)hipFree(places_d);
        if (status_d) (void)hipFree(status_d);
        if (guv) (void)hipFree(guv);
        if (seed_cdl) (void)hipFree(seed_cdl);
        if (stream) (void)hipStreamDestroy(stream);
    }
};

namespace {

void ensure_tables(exaca_ensemble *e, const exaca::HostDomain &h, const std::string &orientation_file) {
    using namespace exaca;
    if (e->guv) {
        if (orientation_file != e->orientation_file)
            throw std::invalid_argument("all domains of an ensemble share one orientation file");
        return;
    }
    e->orientation_file = orientation_file;
    const std::vector<float> seed = seed_table(h.guv, kNumOrientations);
    HIP_OK(hipMalloc(&e->guv, h.guv.size() * 4));
    HIP_OK(hipMalloc(&e->seed_cdl, seed.size() * 4));
    HIP_OK(hipMemcpy(e->guv, h.guv.data(), h.guv.size() * 4, hipMemcpyHostToDevice));
    HIP_OK(hipMemcpy(e->seed_cdl, seed.data(), seed.size() * 4, hipMemcpyHostToDevice));
}

// Estimated time of a step (us) of a domain with that cross-section and team: a chain that grows
// with the team's barriers, and the front's cells by the team, dearer in a large domain, whose records
// the caches don't hold. Single domains measured, us: 24^3 7.1
// with 1 workgroup, 44^3 17.7 with 1 and 13.4 with 8, 100^3 138 with 1, 27.6 with 8 and 18.7 with 32, 150^3 54.0
// with 8 and 22.9 with 64.
double step_estimate(const exaca::DomainView &d, int team) {
    const double chain = team == 1 ? 3.0 : 7.0 + std::log2(static_cast<double>(team));
    const double per_cell = 0.0075 + 0.0125 * std::min(1.0, static_cast<double>(d.ncell) / 1.6e7);
    return chain + per_cell * static_cast<double>(d.X) * d.Y / team;
}

// The workgroups of a launch. A launch lasts as long as its slowest domain, and no less than all
// domains' workgroup time over the device's CUs (a workgroup takes a CU; those that find none wait for
// the domains before them to finish their steps). Every running domain starts with a team of one, and
// the slowest one's team is doubled, up to the workgroups-per-slot setting, while CUs are spare and
// it gains from it; beyond the CUs only while it would take half as long again as its share of them
// (its larger team costs the others time). The largest teams come first, so that the small domains
// fill in behind them. Measured, ms for all solves (at most 32 workgroups a slot) within the CUs only,
// beyond them with a factor of 2, this 1.5, 1.1 and 1: 256 domains of sides 32-256 3562, 2380, 2094, 1918, 1963;
// 256 of 32-64 203, 203, 204, 216, 216; 64 of 32-64 92, 92, 92, 104, 110; 16 of 64-192 185, 184, 185, 184, 192.
void share_out(exaca_ensemble *e) {
    if (!e->dirty) return;
    std::vector<std::pair<double, int>> running;  // estimate, slot
    std::vector<int> team(e->slots, 0);
    double area = 0;  // workgroup time of all
    int total = 0;    // workgroups
    for (int s = 0; s < e->slots; s++)
        if (e->used[s] && e->status[s] == 0) {
            team[s] = 1;
            running.emplace_back(step_estimate(e->views[s], 1), s);
            area += running.back().first;
            total++;
        }
    const int most = std::min(e->blocks, exaca::kMaxTeam);
    std::make_heap(running.begin(), running.end());
    while (!running.empty()) {
        std::pop_heap(running.begin(), running.end());
        const auto [t, s] = running.back();
        running.pop_back();
        if (2 * team[s] > most) break;
        const double less = step_estimate(e->views[s], 2 * team[s]);
        const double grown = area + 2 * team[s] * less - team[s] * t;
        if (less > 0.95 * t) break;  // the slowest domain gains nothing from more
        if (total + team[s] > e->cus && t < 1.5 * grown / e->cus) break;
        area = grown;
        total += team[s];
        team[s] *= 2;
        running.emplace_back(less, s);
        std::push_heap(running.begin(), running.end());
    }
    e->places.clear();
    for (int nb = exaca::kMaxTeam; nb >= 1; nb /= 2)
        for (int s = 0; s < e->slots; s++)
            if (team[s] == nb)
                for (int b = 0; b < nb; b++)
                    e->places.push_back(exaca::TeamPlace{static_cast<uint32_t>(s), static_cast<uint32_t>(b),
                                                         static_cast<uint32_t>(nb)});
    if (!e->places.empty()) {
        if (e->places.size() > e->places_cap) {
            HIP_OK(hipStreamSynchronize(e->stream));
            if (e->places_d) HIP_OK(hipFree(e->places_d));
            e->places_d = nullptr;
            e->places_cap = 0;
            HIP_OK(hipMalloc(&e->places_d, sizeof(exaca::TeamPlace) * 2 * e->places.size()));
            e->places_cap = 2 * e->places.size();
        }
        HIP_OK(hipMemcpyAsync(e->places_d, e->places.data(), sizeof(exaca::TeamPlace) * e->places.size(),
                              hipMemcpyHostToDevice, e->stream));
        HIP_OK(hipStreamSynchronize(e->stream));  // e->places may change
    }
    e->dirty = false;
}

// Enqueues `steps` steps (a multiple of kChunk) of every running domain.
void launch(exaca_ensemble *e, int steps) {
    share_out(e);
    e->steps += steps;
    if (e->places.empty()) return;
    for (int n; steps > 0; steps -= n) {
        n = std::min(steps, kMaxLaunch);
        exaca::launch_steps_n(e->views_d, e->places_d, static_cast<uint32_t>(e->places.size()), n, 0, ++e->launches,
                              e->stream);
        HIP_OK(hipGetLastError());
    }
}

void admit(exaca_ensemble *e, const exaca_prepared *pr, int *slot_out) {
    using namespace exaca;
    ensure_tables(e, pr->host, pr->deck.orientation_file);
    const uint32_t stage = exaca::claim_stage();  // refused before anything is taken
    int slot = -1;
    for (int s = 0; s < e->slots; s++)
        if (!e->used[s]) {
            slot = s;
            break;
        }
    if (slot < 0) throw StateError("no free slot");
    size_t off = 0;
    if (!e->arena.take(pr->bytes, off)) throw StateError("device memory budget exhausted");
    const HostDomain &hd = pr->host;
    const size_t n = static_cast<size_t>(hd.ncell);
    char *p = e->arena.base + off;
    auto carve = [&](size_t bytes) {
        char *q = p;
        p += up(bytes);
        return q;
    };
    std::vector<int32_t> loc, time;
    exaca::layer_sites(hd, 0, loc, time);
    DomainView d{};
    exaca::set_geometry(d, hd.X, hd.Y, hd.nz, hd.nzA);
    d.xoff = hd.xoff;
    d.yoff = hd.yoff;
    d.cells = reinterpret_cast<Cell *>(carve(sizeof(Cell) * n));
    d.octa = reinterpret_cast<Octa *>(carve(sizeof(Octa) * n));
    d.claim_cell = reinterpret_cast<uint32_t *>(carve(4 * exaca::claim_entries(d, exaca::kMaxTeam)));
    d.claim_bits = reinterpret_cast<uint32_t *>(carve(4 * exaca::claim_entries(d, exaca::kMaxTeam)));
    d.sync = reinterpret_cast<uint32_t *>(carve(4 * kSyncWords));
    int32_t *nloc = reinterpret_cast<int32_t *>(carve(4 * std::max<size_t>(hd.nloc.size(), 1)));
    int32_t *ntime = reinterpret_cast<int32_t *>(carve(4 * std::max<size_t>(hd.nloc.size(), 1)));
    double *grow = reinterpret_cast<double *>(carve(8 * pr->grow.size()));
    uint32_t *sums = reinterpret_cast<uint32_t *>(carve(4 * pr->sums.sums.size()));
    d.alarms = reinterpret_cast<uint32_t *>(carve(4 * kAlarmSlots * alarm_stride(d.ncell)));
    d.ctl = reinterpret_cast<StepCtl *>(carve(sizeof(StepCtl)));
    d.stats = reinterpret_cast<StepStats *>(carve(sizeof(StepStats)));
    d.claim_stage = stage;
    d.meet_wait = e->meet_wait;
    d.barrier_wait = e->barrier_wait;
    d.nparts = kMaxTeam;
    d.part = reinterpret_cast<unsigned long long *>(carve(8ull * kPartRows * kMaxTeam));
    d.nnuclei = static_cast<int32_t>(loc.size());
    d.nloc = nloc;
    d.ntime = ntime;
    d.guv = e->guv;
    d.seed_cdl = e->seed_cdl;
    d.grow = grow;
    d.gsat = pr->grow.back();
    d.ksat = pr->ksat;
    d.grow_sums = sums;
    d.sums_usable = pr->sums.usable;
    d.autostop = 1;
    d.liquid0 = pr->liquid0;
    d.status = e->status_d + slot;
    d.status_err = e->status_d + e->slots + slot;

    hipStream_t s = e->stream;
    if (!loc.empty()) {
        HIP_OK(hipMemcpyAsync(nloc, loc.data(), 4 * loc.size(), hipMemcpyHostToDevice, s));
        HIP_OK(hipMemcpyAsync(ntime, time.data(), 4 * time.size(), hipMemcpyHostToDevice, s));
    }
    HIP_OK(hipMemcpyAsync(grow, pr->grow.data(), 8 * pr->grow.size(), hipMemcpyHostToDevice, s));
    HIP_OK(hipMemcpyAsync(sums, pr->sums.sums.data(), 4 * pr->sums.sums.size(), hipMemcpyHostToDevice, s));
    exaca::upload_cells(d, hd, nullptr, s);
    // Chunks end on parity 0, so a new domain always starts in slot 0 of its control block.
    StepCtl c = exaca::initial_ctl(hd);
    HIP_OK(hipMemcpyAsync(d.ctl, &c, sizeof c, hipMemcpyHostToDevice, s));
    HIP_OK(hipMemsetAsync(d.stats, 0, sizeof(StepStats), s));
    HIP_OK(hipMemsetAsync(d.part, 0, 8ull * kPartRows * kMaxTeam, s));
    HIP_OK(hipMemsetAsync(d.sync, 0, 4 * kSyncWords, s));
    const int32_t zero = 0;
    HIP_OK(hipMemcpyAsync(e->status_d + slot, &zero, 4, hipMemcpyHostToDevice, s));
    HIP_OK(hipMemcpyAsync(e->status_d + e->slots + slot, &zero, 4, hipMemcpyHostToDevice, s));
    HIP_OK(hipMemcpyAsync(e->views_d + slot, &d, sizeof d, hipMemcpyHostToDevice, s));
    HIP_OK(hipStreamSynchronize(s));  // the host-side sources above are temporaries
    e->views[slot] = d;
    e->off[slot] = off;
    e->len[slot] = pr->bytes;
    e->used[slot] = 1;
    e->status[slot] = 0;
    e->status[e->slots + slot] = 0;
    e->dirty = true;
    *slot_out = slot;
}

void release(exaca_ensemble *e, int slot) {
    if (slot < 0 || slot >= e->slots || !e->used[slot]) throw std::invalid_argument("slot not in use");
    exaca::DomainView empty{};
    HIP_OK(hipMemcpyAsync(e->views_d + slot, &empty, sizeof empty, hipMemcpyHostToDevice, e->stream));
    HIP_OK(hipStreamSynchronize(e->stream));
    e->arena.give(e->off[slot], e->len[slot]);
    e->views[slot] = empty;
    e->used[slot] = 0;
    e->status[slot] = -1;
    e->status[e->slots + slot] = 0;
    e->dirty = true;
}

void advance(exaca_ensemble *e, int steps) { launch(e, (steps + kChunk - 1) / kChunk * kChunk); }

void poll(exaca_ensemble *e) {
    HIP_OK(hipMemcpyAsync(e->status.data(), e->status_d, 8 * e->slots, hipMemcpyDeviceToHost, e->stream));
    HIP_OK(hipStreamSynchronize(e->stream));
    for (int s = 0; s < e->slots; s++)
        if (!e->used[s]) {
            e->status[s] = -1;
            e->status[e->slots + s] = 0;
        }
    for (const exaca::TeamPlace &p : e->places)
        if (p.b == 0 && e->status[p.slot] != 0) e->dirty = true;  // finished: its workgroups serve the others
}

unsigned long long frontier_total(exaca_ensemble *e) {
    unsigned long long t = 0;
    for (int s = 0; s < e->slots; s++) {
        if (!e->used[s]) continue;
        exaca::StepStats st;
        HIP_OK(hipMemcpy(&st, e->views[s].stats, sizeof st, hipMemcpyDeviceToHost));
        t += st.frontier;
    }
    return t;
}

}  // namespace

extern "C" {

int exaca_prepare(const char *input_file, const char *data_dir, uint64_t seed, exaca_prepared **out) {
    return guarded([&] {
        if (!input_file || !out) throw std::invalid_argument("null argument");
        *out = nullptr;
        auto pr = std::make_unique<exaca_prepared>();
        pr->deck = exaca::read_deck(input_file, data_dir ? data_dir : exaca::data_dir());
        if (pr->deck.sim_type != "C")
            throw std::invalid_argument("ensembles hold directional-solidification (type C) domains");
        pr->deck.seed = seed;
        pr->host = exaca::initialize_sparse(pr->deck, false);
        const exaca::HostDomain &h = pr->host;
        pr->grow = exaca::growth_table(h.A, h.B, h.C, h.D, h.dU, 1 << 25);
        if (pr->grow.size() >= (1u << 25)) throw std::runtime_error("undercooling never saturates within 2^25 steps");
        pr->ksat = exaca::growth_plateau(pr->grow);
        pr->sums = exaca::growth_sums(pr->grow, pr->ksat);
        if (h.ncell > exaca::kEnsembleCells)
            throw std::invalid_argument("domain too large for an ensemble slot (at most " +
                                        std::to_string(exaca::kEnsembleCells) + " cells); run it on the plain path");
        if (h.sparse)  // every cell inside the walls is liquid but the substrate's active cells
            pr->liquid0 = static_cast<long long>(h.nx) * h.ny * (h.nz - 2) - static_cast<long long>(h.active.size());
        else
            for (long long q = 0; q < h.ncell; q++) pr->liquid0 += (h.ct[q] == exaca::kLiquid && h.lid[q] == 0);
        pr->bytes = domain_bytes(h, pr->grow.size(), pr->sums.sums.size());
        *out = pr.release();
    });
}

int exaca_prepared_info(const exaca_prepared *pr, int64_t out[4]) {
    return guarded([&] {
        if (!pr || !out) throw std::invalid_argument("null argument");
        out[0] = pr->host.ncell;
        out[1] = static_cast<int64_t>(pr->bytes);
        out[2] = static_cast<int64_t>(pr->host.nloc.size());
        out[3] = pr->liquid0;
    });
}

int exaca_prepared_free(exaca_prepared *pr) {
    return guarded([&] { delete pr; });
}

int exaca_ensemble_create(int slots, size_t arena_bytes, exaca_ensemble **out) {
    return guarded([&] {
        if (!out || slots <= 0 || slots > 65535 || arena_bytes < kAlign) throw std::invalid_argument("bad argument");
        *out = nullptr;
        auto e = std::make_unique<exaca_ensemble>();
        e->slots = slots;
        e->meet_wait = exaca::meet_wait_ticks();
        e->barrier_wait = exaca::barrier_wait_ticks();
        HIP_OK(hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking));
        HIP_OK(hipMalloc(&e->arena.base, arena_bytes));
        e->arena.bytes = arena_bytes;
        e->arena.free[0] = arena_bytes;
        HIP_OK(hipMalloc(&e->views_d, sizeof(exaca::DomainView) * slots));
        HIP_OK(hipMemset(e->views_d, 0, sizeof(exaca::DomainView) * slots));
        HIP_OK(hipMalloc(&e->status_d, 8 * slots));
        HIP_OK(hipMemset(e->status_d, 0, 8 * slots));
        int dev = 0;
        HIP_OK(hipGetDevice(&dev));
        HIP_OK(hipDeviceGetAttribute(&e->cus, hipDeviceAttributeMultiprocessorCount, dev));
        e->views.assign(slots, exaca::DomainView{});
        e->status.assign(2 * static_cast<size_t>(slots), -1);
        std::fill(e->status.begin() + slots, e->status.end(), 0);
        e->off.assign(slots, 0);
        e->len.assign(slots, 0);
        e->used.assign(slots, 0);
        *out = e.release();
    });
}

int exaca_ensemble_admit(exaca_ensemble *e, const exaca_prepared *pr, int *slot) {
    return guarded([&] {
        if (!e || !pr || !slot) throw std::invalid_argument("null argument");
        admit(e, pr, slot);
    });
}

int exaca_ensemble_release(exaca_ensemble *e, int slot) {
    return guarded([&] {
        if (!e) throw std::invalid_argument("null handle");
        release(e, slot);
    });
}

int exaca_ensemble_advance(exaca_ensemble *e, int steps) {
    return guarded([&] {
        if (!e || steps < 0) throw std::invalid_argument("bad argument");
        advance(e, steps);
    });
}

int exaca_ensemble_poll(exaca_ensemble *e, int32_t *final_cycles, int32_t *errors) {
    return guarded([&] {
        if (!e || !final_cycles) throw std::invalid_argument("null argument");
        poll(e);
        std::copy(e->status.begin(), e->status.begin() + e->slots, final_cycles);
        if (errors) std::copy(e->status.begin() + e->slots, e->status.end(), errors);
    });
}

int exaca_ensemble_set_blocks(exaca_ensemble *e, int blocks) {
    return guarded([&] {
        if (!e || blocks < 8 || blocks > kMaxBlocks || blocks % 8) throw std::invalid_argument("bad workgroup count");
        e->blocks = blocks;
        e->dirty = true;
    });
}

int exaca_ensemble_autotune(exaca_ensemble *e, int chunks_per_candidate, int *chosen) {
    return guarded([&] {
        if (!e || !chosen || chunks_per_candidate <= 0) throw std::invalid_argument("bad argument");
        // Online tuning on the live ensemble: the workgroup count per slot changes only the
        // schedule, never the result, so candidates are tried on consecutive chunks and scored by
        // device time per active-cell update. A team never has more than kMaxTeam workgroups, so larger
        // settings are the same as that one.
        const int candidates[] = {16, 32, exaca::kMaxTeam};
        double best = 1e300;
        int best_b = candidates[0];
        hipEvent_t e0, e1;
        HIP_OK(hipEventCreate(&e0));
        HIP_OK(hipEventCreate(&e1));
        for (int b : candidates) {
            e->blocks = b;
            e->dirty = true;
            share_out(e);
            HIP_OK(hipStreamSynchronize(e->stream));
            const unsigned long long f0 = frontier_total(e);
            HIP_OK(hipEventRecord(e0, e->stream));
            for (int c = 0; c < chunks_per_candidate; c++) launch(e, kChunk);
            HIP_OK(hipEventRecord(e1, e->stream));
            HIP_OK(hipEventSynchronize(e1));
            float ms = 0;
            HIP_OK(hipEventElapsedTime(&ms, e0, e1));
            const unsigned long long f1 = frontier_total(e);
            const double score = ms / static_cast<double>(std::max<unsigned long long>(f1 - f0, 1));
            if (score < best) {
                best = score;
                best_b = b;
            }
        }
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        e->blocks = best_b;
        e->dirty = true;
        *chosen = best_b;
    });
}

int exaca_ensemble_query(exaca_ensemble *e, int slot, int64_t out[8]) {
    return guarded([&] {
        if (!e || !out || slot < 0 || slot >= e->slots || !e->used[slot]) throw std::invalid_argument("bad slot");
        exaca::StepStats st;
        exaca::StepCtl c;
        HIP_OK(hipStreamSynchronize(e->stream));
        HIP_OK(hipMemcpy(&st, e->views[slot].stats, sizeof st, hipMemcpyDeviceToHost));
        HIP_OK(hipMemcpy(&c, e->views[slot].ctl, sizeof c, hipMemcpyDeviceToHost));
        out[0] = c.done ? c.final_cycle : 0;
        out[1] = static_cast<int64_t>(st.nucleated);
        out[2] = static_cast<int64_t>(st.frontier);
        out[3] = static_cast<int64_t>(st.captures);
        out[4] = static_cast<int64_t>(st.solidified);
        out[5] = c.error;
        out[6] = static_cast<int64_t>(e->arena.available());
        out[7] = e->steps;
    });
}

int exaca_ensemble_download(exaca_ensemble *e, int slot, int field, void *dst, size_t dst_bytes) {
    return guarded([&] {
        if (!e || !dst || slot < 0 || slot >= e->slots || !e->used[slot]) throw std::invalid_argument("bad slot");
        exaca::download_field(e->views[slot], field, dst, dst_bytes, e->stream);
    });
}

int exaca_ensemble_destroy(exaca_ensemble *e) {
    return guarded([&] { delete e; });
}

}  // extern "C"
