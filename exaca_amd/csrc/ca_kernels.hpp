// ca_kernels.hpp -- host-side launchers for the CDNA4 kernels of one CA time step.
#pragma once
#include <hip/hip_runtime.h>

#include "ca_common.hpp"

namespace exaca {

constexpr int kBlock = 256;  // four wave64s per workgroup

// A step as its kernels are told of it: the cycle, the steps executed before it, whether the step before
// ran just before it (no cycle jump, same layer), and its parity in the control block.
struct StepAt {
    int cycle;
    uint32_t serial;
    int follows, parity;
};
// Nucleation (src/CAupdate.cpp:67-200). A step may leave it out when no site's time falls in the
// steps since nucleation last ran (it would examine nothing).
void launch_nucleation(const DomainView &d, const StepAt &at, hipStream_t s);
// Its workgroups (each adds to its own slot of the nucleation counter rows).
int nucleation_blocks(const DomainView &d);
// CellCapture (src/CAupdate.cpp:204-728) in two kernels: the liquidus-time gate, growth, neighbour
// scan and claims of the cells due this step (also prepares the control slot of the next step);
// then claims decided and winners' captures.
void launch_capture(const DomainView &d, const StepAt &at, int blocks, hipStream_t s);
// The solidifications the last step left to the next one, and the counters booked: before the state
// or the statistics are looked at. parity_next is the parity of the next step.
void launch_settle(const DomainView &d, int parity_next, int blocks, hipStream_t s);
// `steps` steps in one launch of a team of workgroups (at most kMaxTeam), settled and booked;
// nucleate: with their nucleation (else none of their sites may be due). launch: a number greater than 0 and
// those of the domain's launches before.
constexpr int kTeamBlock = 512;
void launch_steps(const DomainView &d, int parity, int layer, int steps, bool nucleate, int team, uint64_t launch,
                  hipStream_t s);
// Capture-pass workgroups that a CU holds at once.
int claim_per_cu();
// Entries of the claim lists for up to most_blocks capture-pass workgroups.
size_t claim_entries(const DomainView &d, uint32_t most_blocks);
// Every active cell due at the next step: after a cycle jump, whose skipped steps the calendar did
// not count. parity_next is the parity of the next step.
void launch_rewake(const DomainView &d, int parity_next, int blocks, hipStream_t s);
// The next layer's window: out[0] = least z of an active cell, out[1] = greatest z of a cell of
// next_layer (out initialised to INT32_MAX, -1 by the caller).
void launch_layer_bounds(const DomainView &d, int next_layer, int *out, hipStream_t s);
// LayerSetup on the resident state for the window [d.zlo, d.nzA).
void launch_layer_setup(const DomainView &d, int parity_next, hipStream_t s);
// `steps` steps (an even number, from parity 0) of the domains of a device-resident table of views,
// settled and booked: one workgroup per entry of `places`.
void launch_steps_n(const DomainView *views, const TeamPlace *places, uint32_t workgroups, int steps, int layer,
                    uint64_t launch, hipStream_t s);
// IntermediateOutputAndCheck's reduction (src/CAupdate.cpp:738-758, 792-808).
void launch_check(const DomainView &d, int cycle, int layer, CheckResult *out, hipStream_t s);
// Octahedra of the initially active cells (src/CAinitialize.cpp:1936-2043).
void launch_seed_init(const DomainView &d, const uint32_t *cells, uint32_t n, hipStream_t s);
// One step with an event pair around each kernel: nucleation, claim and apply. ev holds
// 2 * kTimedKernels events.
constexpr int kTimedKernels = 3;
void launch_step_timed(const DomainView &d, const StepAt &at, int blocks, hipStream_t s, hipEvent_t *ev);
// Initial cell records from compact device arrays (CellType with the seed bit, LayerID, GrainID,
// CritTimeStep), and one field back out of the records (FieldKind layout).
void launch_pack(const DomainView &d, const uint8_t *ct, const int8_t *lid, const int32_t *gid, const int32_t *cts,
                 hipStream_t s);
void launch_extract(const DomainView &d, int field, void *out, hipStream_t s);
// The initial state of a directional-solidification domain built on the device from its per-plane
// CritTimeStep, the substrate's active cells and the nucleation sites (both in index order); the
// Melted flags go to `melted` (one byte per cell).
void launch_init_directional(const DomainView &d, const int32_t *plane_cts, int nx, int ny, uint8_t *melted,
                             const uint32_t *substrate, uint32_t nsub, const int32_t *sites, uint32_t nsites,
                             hipStream_t s);
// Bytes per cell of a field as launch_extract writes it (0: not a per-cell field).
inline size_t field_bytes(int field) {
    switch (field) {
    case kFieldCellTypeRaw: return 1;
    case kFieldCentre: return 12;
    case kFieldCentreF64: return 24;
    case kFieldCellType:
    case kFieldGrainId:
    case kFieldDiagonal:
    case kFieldCritTimeStep:
    case kFieldLayerId: return 4;
    default: return 0;
    }
}
// Grain statistics of the whole-domain region [k0, k1] x [i0, i1] x [j0, j1] (inclusive; the
// reference's vtk / analysis layout): flags gflag[GrainID - gmin] (ngid entries), counts[0..2] +=
// melted cells, cells with a negative GrainID, cells whose GrainID falls outside the flag range;
// obins / otop += melted cells per orientation, in the region / in its top plane k1.
struct GrainRegion {
    int k0, k1, i0, i1, j0, j1;
};
void launch_grain_stats(const DomainView &d, const uint8_t *melted, const GrainRegion &r, int gmin, uint32_t ngid,
                        uint32_t *gflag, unsigned long long *counts, unsigned int *obins, unsigned int *otop,
                        hipStream_t s);
// The largest ensemble domain.
constexpr long long kEnsembleCells = 1ll << 25;
// Unique GrainIDs of a grain-statistics pass: the nonzero entries of gflag[0..n), added to *out.
void launch_count_flags(const uint32_t *gflag, uint32_t n, unsigned long long *out, hipStream_t s);
// The cells due at the step of that serial, added to *out.
void launch_count_due(const DomainView &d, uint32_t serial, unsigned long long *out, hipStream_t s);
// p[0..n) = v, as a kernel (no memset node in a captured graph).
void launch_fill(uint32_t *p, size_t n, uint32_t v, hipStream_t s);
// Plain copy of n 16-byte words (HBM calibration).
void launch_copy(const uint4 *src, uint4 *dst, size_t n, hipStream_t s);
// Device-side self test of the capture geometry against host values: one octahedron per input row.
void launch_geometry_probe(const float *guv, const double *in, double *out, int n, hipStream_t s);

}  // namespace exaca
