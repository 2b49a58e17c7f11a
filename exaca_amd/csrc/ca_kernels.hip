// ca_kernels.hip -- the CA time step as memory-bound CDNA4 kernels over the cells due this step.
//
// One step (reference: src/runCA.cpp:291-311) is two launches on one stream (three when a nucleation
// site can be due):
//   k_nucleate  activates the pre-sampled nuclei whose time has come (src/CAupdate.cpp:67-200)
//   k_claim     for every cell due this step, gathered from the step's calendar slot: the growth
//               since it was last looked at, a claim on every liquid neighbour it reaches (atomicMin
//               of its index into the neighbour's claim word), and the step at which it is due next;
//               a cell past its liquidus time with no liquid neighbour turns solid
//   k_apply     the claimants that won a claim (their index is in the claimed cell's word) capture:
//               each builds the new decentred octahedron, stores its 26 critical lengths, and takes
//               the cell out of its neighbours' liquid masks
// A cell whose liquid neighbours were all taken by lower-indexed cells in a step turns solid in that
// step: the claim pass of the next step finds it due and gives it that step's state, and k_settle does
// so when the caller looks at the state in between; k_book then sums the steps' counters.
// What bounds a step of all but the widest domains is not its work but what a launch costs before and
// between its loads (5-14 us a kernel for a few dozen cells: caches and code are cold after each kernel
// boundary), so a step has as few phases as its domain-wide dependences allow: claims before winners,
// captures before the next step's claims. With separate kernels for the winners, the settling and the
// list of due cells a step took 28.8, 40.5, 66.4, 76.4 us at 24^3, 100^3, 256^3, 400^3; with two kernels
// it takes 12.1, 15.9, 25.2, 36.4 us; at 800^3 (cycles 6006-6025) 0.198 and 0.155 ms.
// A narrow domain takes its steps in k_steps, many in a launch: a team of 1 to 64 workgroups with a
// barrier between the phases of a step (6.9 us a step at 24^3, 15.5 at 100^3); k_steps_n does so for
// every domain of an ensemble.
// A cell is due when something can happen to it: it is new, its liquidus time has passed, or its
// half-diagonal reaches the least critical length of its liquid neighbours; a neighbour's capture
// or nucleation that empties its mask is handled where it happens. Between those steps its growth
// is a fixed recurrence, applied exactly when it is next looked at.
// Claim-then-apply reproduces the reference's Serial backend exactly: there pass 2 visits active
// cells in ascending index order and every capture is visible at once, so a liquid cell goes to
// the lowest-indexed cell that reaches it, and cell j still "sees" a liquid neighbour only if no
// lower-indexed cell took it (src/CAupdate.cpp:264-352, 722-725).
//
// Every floating-point expression keeps the reference's operation order and float/double types;
// the library is compiled with -ffp-contract=off and correctly rounded fp32 divide/sqrt.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "ca_kernels.hpp"
#include "growth.hpp"
#include "meet.hpp"
#include "threshold.hpp"

namespace exaca {
namespace {

__device__ __forceinline__ double dmin(double a, double b) { return (b < a) ? b : a; }  // std::min
__device__ __forceinline__ double dmax(double a, double b) { return (a < b) ? b : a; }  // std::max

__device__ __forceinline__ int orientation_of(int gid) { return (abs(gid) - 1) % kNumOrientations; }

// Steps executed in (t, cycle] of one layer whose cycle jumps are entries j0 .. j1-1: the reference
// adds the undercooling change once per executed step while a cell is liquid or active past its
// liquidus time (src/CAupdate.cpp:235-237); cycle jumps (src/CAupdate.cpp:812-814) skip steps
// J+1 .. T-1.
__device__ __forceinline__ int executed_in(int t, int cycle, const StepCtl *ctl, int j0, int j1) {
    int n = cycle - t;
    for (int q = j0; q < j1; q++) {
        const int lo = max(ctl->jump_from[q] + 1, t + 1);
        const int hi = min(ctl->jump_to[q] - 1, cycle);
        if (hi >= lo) n -= hi - lo + 1;
    }
    return n;
}

struct Coord {
    int x, y, z;
};
// Offsets of neighbour l (a per-lane value) decoded from the packed constants.
__device__ __forceinline__ int nb_dx(int l) { return static_cast<int>((kPackX >> (2 * l)) & 3u) - 1; }
__device__ __forceinline__ int nb_dy(int l) { return static_cast<int>((kPackY >> (2 * l)) & 3u) - 1; }
__device__ __forceinline__ int nb_dz(int l) { return static_cast<int>((kPackZ >> (2 * l)) & 3u) - 1; }

struct Grid {
    Divisor xy, y;
    int X, Y, nzA;
    int row[9];  // linear offsets of the rows of neighbours, (dz + 1) * 3 + dx + 1
    // linear offset of neighbour l for a per-lane l
    __device__ __forceinline__ int offset(int l) const {
        return nb_dz(l) * static_cast<int>(xy.d) + nb_dx(l) * Y + nb_dy(l);
    }
};
__device__ __forceinline__ Grid grid_of(const DomainView &d) {
    Grid g;
    g.X = d.X;
    g.Y = d.Y;
    g.nzA = d.nzA;
    g.xy = d.by_xy;
    g.y = d.by_y;
#pragma unroll
    for (int r = 0; r < 9; r++) g.row[r] = ((r / 3 - 1) * d.X + (r % 3 - 1)) * d.Y;
    return g;
}
// The neighbours of cell q by rows: neighbour l is one of three consecutive cells of a row, so the
// nine row addresses and constant offsets reach all 26 (26 addresses of their own would cost the
// capture pass 34 more registers).
struct Rows {
    Cell *row[9];
    __device__ __forceinline__ Cell &cell(int l) const { return row[(kNbZ[l] + 1) * 3 + kNbX[l] + 1][kNbY[l]]; }
    // the low word of a cell's liquid-neighbour mask (bits 0-25 and the not-yet-known bit), and the high word
    __device__ __forceinline__ uint32_t *low(int l) const { return reinterpret_cast<uint32_t *>(&cell(l).lm); }
    __device__ __forceinline__ uint32_t *high(int l) const { return low(l) + 1; }
};
// A cell that is active or was liquid lies inside the walls, so all 26 of its linear neighbours lie
// in the array: they can be read without a test each, and masked by the valid ones after. For a cell
// that did not (there is none), the nearest one that does, and no valid neighbour.
__device__ __forceinline__ uint32_t inner_cell(const DomainView &d, const Grid &g, uint32_t q, uint32_t &valid) {
    const uint32_t reach = g.xy.d + g.y.d + 1, last = static_cast<uint32_t>(d.ncell) - 1 - reach;
    const uint32_t at = q < reach ? reach : (q > last ? last : q);
    valid = at == q ? valid : 0u;
    return at;
}
__device__ __forceinline__ Rows rows_of(const DomainView &d, const Grid &g, uint32_t q, uint32_t &valid) {
    const uint32_t at = inner_cell(d, g, q, valid);
    Rows r;
#pragma unroll
    for (int i = 0; i < 9; i++) r.row[i] = d.cells + static_cast<uint32_t>(at + g.row[i]);
    return r;
}
__device__ __forceinline__ Coord decode(uint32_t p, const Grid &g) {
    Coord c;
    const uint32_t z = g.xy.div(p);
    const uint32_t rem = p - z * g.xy.d;
    const uint32_t x = g.y.div(rem);
    c.z = static_cast<int>(z);
    c.x = static_cast<int>(x);
    c.y = static_cast<int>(rem - x * g.y.d);
    return c;
}
__device__ __forceinline__ Coord decode(uint32_t p, int X, int Y) {
    const uint32_t XY = static_cast<uint32_t>(X) * static_cast<uint32_t>(Y);
    Coord c;
    c.z = static_cast<int>(p / XY);
    const uint32_t rem = p - static_cast<uint32_t>(c.z) * XY;
    c.x = static_cast<int>(rem / static_cast<uint32_t>(Y));
    c.y = static_cast<int>(rem - static_cast<uint32_t>(c.x) * static_cast<uint32_t>(Y));
    return c;
}
// Neighbours inside the rank's slab and below the active-domain top; the reference's edge lists
// (src/CAupdate.cpp:276-318) and its MyNeighborZ < nzActive test (:328). z >= 0 always holds for
// an active cell (plane 0 is a wall); it is tested for memory safety.
__device__ __forceinline__ uint32_t valid_neighbours(const Coord &c, int X, int Y, int nzA) {
    if (c.x > 0 && c.x < X - 1 && c.y > 0 && c.y < Y - 1 && c.z > 0 && c.z < nzA - 1) return (1u << 26) - 1;
    uint32_t m = 0;
#pragma unroll
    for (int l = 0; l < 26; l++) {
        const int x = c.x + kNbX[l], y = c.y + kNbY[l], z = c.z + kNbZ[l];
        if (x >= 0 && x < X && y >= 0 && y < Y && z >= 0 && z < nzA) m |= 1u << l;
    }
    return m;
}

// Face normals of the octahedron as the reference forms them: float sums of unit-vector
// components (src/CAupdate.cpp:526-551).
struct Faces {
    double fx[4], fy[4], fz[4];
};
__device__ __forceinline__ Faces faces_of(const float *g) {
    Faces f;
    f.fx[0] = g[0] + g[3] + g[6];
    f.fx[1] = g[0] - g[3] + g[6];
    f.fx[2] = g[0] + g[3] - g[6];
    f.fx[3] = g[0] - g[3] - g[6];
    f.fy[0] = g[1] + g[4] + g[7];
    f.fy[1] = g[1] - g[4] + g[7];
    f.fy[2] = g[1] + g[4] - g[7];
    f.fy[3] = g[1] - g[4] - g[7];
    f.fz[0] = g[2] + g[5] + g[8];
    f.fz[1] = g[2] - g[5] + g[8];
    f.fz[2] = g[2] + g[5] - g[8];
    f.fz[3] = g[2] - g[5] - g[8];
    return f;
}
// Critical diagonal length of neighbour l for an octahedron centred at c around the cell centre
// (xp, yp, zp): the largest |F_q . (x_l - c)| (src/CAupdate.cpp:553-563), rounded to float as
// the reference stores it.
__device__ __forceinline__ float critical_length(const Faces &f, double xp, double yp, double zp, double cx,
                                                 double cy, double cz, int dx, int dy, int dz) {
    const double ex = xp + dx - cx, ey = yp + dy - cy, ez = zp + dz - cz;
    const double d0 = ex * f.fx[0] + ey * f.fy[0] + ez * f.fz[0];
    const double d1 = ex * f.fx[1] + ey * f.fy[1] + ez * f.fz[1];
    const double d2 = ex * f.fx[2] + ey * f.fy[2] + ez * f.fz[2];
    const double d3 = ex * f.fx[3] + ey * f.fy[3] + ez * f.fz[3];
    return static_cast<float>(dmax(dmax(fabs(d0), fabs(d1)), dmax(fabs(d2), fabs(d3))));
}

// The centre of cell q's octahedron record (the last 24 bytes of its line).
__device__ __forceinline__ void set_centre(const DomainView &d, uint32_t q, double x, double y, double z) {
    Octa &o = d.octa[q];
    o.x = x;
    o.y = y;
    o.z = z;
}

struct Octahedron {
    double cx, cy, cz, dl;
};
__device__ __forceinline__ double sel3(int i, double a, double b, double c) { return i == 0 ? a : (i == 1 ? b : c); }

// The captured cell's decentred octahedron (src/CAupdate.cpp:360-515): the capturing face is
// found from the signs of the unit-vector projections, the face corner nearest the new cell
// centre is the new octahedron's tip, and its half-diagonal follows from the projections of the
// centre onto the two face edges through that corner.
__device__ Octahedron new_octahedron(const float *g, double cxold, double cyold, double czold, double xp, double yp,
                                     double zp) {
    const double x0 = xp - cxold, y0 = yp - cyold, z0 = zp - czold;
    // the reference divides these by the distance of the centres; only their signs are used, and
    // the quotient's sign is the dividend's
    const double a1 = g[0] * x0 + g[1] * y0 + g[2] * z0;
    const double a2 = g[3] * x0 + g[4] * y0 + g[5] * z0;
    const double a3 = g[6] * x0 + g[7] * y0 + g[8] * z0;
    const float s1 = (a1 < 0) ? 1.0f : -1.0f, s2 = (a2 < 0) ? 1.0f : -1.0f, s3 = (a3 < 0) ? 1.0f : -1.0f;
    const double d1x = g[0] * s1, d1y = g[1] * s1, d1z = g[2] * s1;
    const double d2x = g[3] * s2, d2y = g[4] * s2, d2z = g[5] * s2;
    const double d3x = g[6] * s3, d3y = g[7] * s3, d3z = g[8] * s3;
    const double u10 = d2x - d1x, u11 = d2y - d1y, u12 = d2z - d1z;
    const double u20 = d3x - d1x, u21 = d3y - d1y, u22 = d3z - d1z;
    const double uu0 = u11 * u22 - u12 * u21, uu1 = u12 * u20 - u10 * u22, uu2 = u10 * u21 - u11 * u20;
    const double nd = sqrtf(static_cast<float>(uu0 * uu0 + uu1 * uu1 + uu2 * uu2));
    const double n0 = uu0 / nd, n1 = uu1 / nd, n2 = uu2 / nd;
    const double t = (n0 * x0 + n1 * y0 + n2 * z0) / (n0 * d1x + n1 * d1y + n2 * d1z);
    const double tx0 = cxold + t * d1x, ty0 = cyold + t * d1y, tz0 = czold + t * d1z;
    const double tx1 = cxold + t * d2x, ty1 = cyold + t * d2y, tz1 = czold + t * d2z;
    const double tx2 = cxold + t * d3x, ty2 = cyold + t * d3y, tz2 = czold + t * d3z;
    const double dc0 = sqrtf(static_cast<float>(((tx0 - xp) * (tx0 - xp)) + ((ty0 - yp) * (ty0 - yp)) +
                                                ((tz0 - zp) * (tz0 - zp))));
    const double dc1 = sqrtf(static_cast<float>(((tx1 - xp) * (tx1 - xp)) + ((ty1 - yp) * (ty1 - yp)) +
                                                ((tz1 - zp) * (tz1 - zp))));
    const double dc2 = sqrtf(static_cast<float>(((tx2 - xp) * (tx2 - xp)) + ((ty2 - yp) * (ty2 - yp)) +
                                                ((tz2 - zp) * (tz2 - zp))));
    const int bx = dc0 < dc1, by = dc1 < dc2, bz = dc2 < dc0;
    const int idx = 2 * (bz - by) * bz + (by - bx) * by;
    const int i1 = (idx + 1) % 3, i2 = (idx + 2) % 3;
    const double mind = sel3(idx, dc0, dc1, dc2);
    const double xc = sel3(idx, tx0, tx1, tx2), yc = sel3(idx, ty0, ty1, ty2), zc = sel3(idx, tz0, tz1, tz2);
    const double x1 = sel3(i1, tx0, tx1, tx2), y1 = sel3(i1, ty0, ty1, ty2), z1 = sel3(i1, tz0, tz1, tz2);
    const double x2 = sel3(i2, tx0, tx1, tx2), y2 = sel3(i2, ty0, ty1, ty2), z2 = sel3(i2, tz0, tz1, tz2);
    const double D1 =
        sqrtf(static_cast<float>(((xp - x2) * (xp - x2)) + ((yp - y2) * (yp - y2)) + ((zp - z2) * (zp - z2))));
    const double D2 =
        sqrtf(static_cast<float>(((xc - x2) * (xc - x2)) + ((yc - y2) * (yc - y2)) + ((zc - z2) * (zc - z2))));
    const double D3 =
        sqrtf(static_cast<float>(((xp - x1) * (xp - x1)) + ((yp - y1) * (yp - y1)) + ((zp - z1) * (zp - z1))));
    const double D4 =
        sqrtf(static_cast<float>(((xc - x1) * (xc - x1)) + ((yc - y1) * (yc - y1)) + ((zc - z1) * (zc - z1))));
    double I1 = 0, I2 = D2, J1 = 0, J2 = D4;
    if (mind != 0) {
        I1 = D1 * ((xp - x2) * (xc - x2) + (yp - y2) * (yc - y2) + (zp - z2) * (zc - z2)) / (D1 * D2);
        I2 = D2 - I1;
        J1 = D3 * ((xp - x1) * (xc - x1) + (yp - y1) * (yc - y1) + (zp - z1) * (zc - z1)) / (D3 * D4);
        J2 = D4 - J1;
    }
    const double sqrt3 = sqrt(3.0);
    const double L12 = 0.5 * (dmin(I1, sqrt3) + dmin(I2, sqrt3));
    const double L13 = 0.5 * (dmin(J1, sqrt3) + dmin(J2, sqrt3));
    const double newdl = sqrt(2.0) * dmax(L12, L13);
    const double c0 = xc - cxold, c1 = yc - cyold, c2 = zc - czold;
    const double cn = sqrt(c0 * c0 + c1 * c1 + c2 * c2);
    Octahedron o;
    o.cx = xc - newdl * (c0 / cn);
    o.cy = yc - newdl * (c1 / cn);
    o.cz = zc - newdl * (c2 / cn);
    o.dl = newdl;
    return o;
}

// Wave64 inclusive prefix sum of v in registers (DPP row shifts and row broadcasts); total is the
// wave sum. Every lane of the wave must reach the call.
__device__ __forceinline__ uint32_t wave_inclusive_scan(uint32_t v, uint32_t &total) {
    int x = static_cast<int>(v);
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);  // row_shr:1
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);  // row_shr:2
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);  // row_shr:4
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);  // row_shr:8
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
    total = static_cast<uint32_t>(__builtin_amdgcn_readlane(x, 63));
    return static_cast<uint32_t>(x);
}

// Wave64 maximum of v, in lane 63 (the same steps; 0 where a lane has no source).
__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
    auto step = [&](int x) { v = static_cast<uint32_t>(x) > v ? static_cast<uint32_t>(x) : v; };
    step(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x111, 0xf, 0xf, false));
    step(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x112, 0xf, 0xf, false));
    step(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x114, 0xf, 0xf, false));
    step(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x118, 0xf, 0xf, false));
    step(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x142, 0xa, 0xf, false));
    step(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x143, 0xc, 0xf, false));
    return v;
}

__device__ __forceinline__ unsigned long long block_sum(unsigned long long v, unsigned long long *sh) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    __syncthreads();
    if (lane == 0) sh[w] = v;
    __syncthreads();
    unsigned long long t = 0;
    if (threadIdx.x == 0)
        for (int q = 0; q < kBlock / 64; q++) t += sh[q];
    return t;
}

// Wave-aggregated append: every lane with `want` gets its own slot of the list behind `counter`
// (LDS), at one atomic per wave. Every lane of the wave must reach the call.
__device__ __forceinline__ uint32_t wave_append(bool want, uint32_t *counter) {
    const unsigned long long b = __ballot(want);
    if (b == 0) return 0;
    const int lane = threadIdx.x & 63;
    const int leader = __ffsll(static_cast<long long>(b)) - 1;
    uint32_t base = 0;
    if (lane == leader) base = atomicAdd(counter, static_cast<uint32_t>(__popcll(b)));
    base = __shfl(base, leader, 64);
    return base + static_cast<uint32_t>(__popcll(b & ((1ull << lane) - 1)));
}

// A cell record read as two 16-byte loads (one 32-byte sector).
struct CellWords {
    unsigned long long lm;
    float dl, thr;
    int32_t cts, gid;
    uint32_t win;
    int8_t lid;
    uint8_t ct;
    uint16_t flags;
};
__device__ __forceinline__ CellWords load_cell(const Cell *c) {
    const uint4 a = reinterpret_cast<const uint4 *>(c)[0];
    const uint4 b = reinterpret_cast<const uint4 *>(c)[1];
    CellWords w;
    w.lm = static_cast<unsigned long long>(a.x) | (static_cast<unsigned long long>(a.y) << 32);
    w.dl = __uint_as_float(a.z);
    w.thr = __uint_as_float(a.w);
    w.cts = static_cast<int32_t>(b.x);
    w.gid = static_cast<int32_t>(b.y);
    w.win = b.z;
    w.lid = static_cast<int8_t>(b.w & 0xFFu);
    w.ct = static_cast<uint8_t>((b.w >> 8) & 0xFFu);
    w.flags = static_cast<uint16_t>(b.w >> 16);
    return w;
}

// The high word of an active cell: serial + 1 of the last step in which a capture by a cell of index
// >= q took one of q's liquid neighbours (0: none yet). Written by the capture pass only where the low
// word is known, so the 64-bit stores of a mask build (which clear it) never meet it in one step.
constexpr uint32_t kMaskUnknown = static_cast<uint32_t>(kLmUnknown);
constexpr uint32_t kMaskNow = static_cast<uint32_t>(kLmNow);
// A liquid cell's words: the low word keeps bits 26-31 of its initial all-ones value (only bits
// 0-25 are ever cleared, by nucleation), bit 30 marking it liquid; the high word is its claim word:
// the lowest index of a cell that claimed it in the current step (kClaimNone: none). A claimed
// cell is captured in the same step and never turns liquid again, so a claim word is read only in
// the step that wrote it, and the capture overwrites both words.
constexpr uint32_t kLiquidMark = 1u << 30;
__device__ __forceinline__ uint32_t *claim_word(const DomainView &d, uint32_t q) {
    return reinterpret_cast<uint32_t *>(&d.cells[q].lm) + 1;
}
__device__ __forceinline__ bool is_unclaimed_liquid(unsigned long long lm) {
    return (static_cast<uint32_t>(lm) & kLiquidMark) && static_cast<uint32_t>(lm >> 32) == kClaimNone;
}

// ---- Growth between events. A cell's half-diagonal grows by grow[k] at the k-th executed step
// past its liquidus time (src/CAupdate.cpp:257-261). Between two events of a cell the growth is
// this fixed recurrence, so it is applied when the cell is next looked at, one float rounding per
// step exactly as the reference stores it. ----

// k of the step at `cycle` of the current layer for cell q: the steps executed past its liquidus
// time in every layer from its own LayerID on in which it lay inside that layer's active window
// (pass 1 visits the window only and accumulates only while LayerID <= layer, and the undercooling
// is never reset between layers; src/CAupdate.cpp:217-237, src/runCA.cpp:283-418). 0 while the cell
// waits for its liquidus time or its layer.
// The layer and its cycle jumps.
struct LayerAt {
    int layer, j0, j1;
};
__device__ __forceinline__ LayerAt layer_at(const DomainView &d) { return LayerAt{d.layer, d.jump0, d.njumps}; }
__device__ __forceinline__ int growth_index(const DomainView &d, const LayerAt &at, int cts, int lid, uint32_t q, int cycle) {
    const StepCtl *c = d.ctl;
    if (lid > at.layer) return 0;
    int k = executed_in(cts, cycle, c, at.j0, at.j1);
    k = k < 0 ? 0 : k;
    const int first = lid < 0 ? 0 : lid;
    if (first < at.layer) {
        const int z = static_cast<int>(d.by_xy.div(q));
        for (int l = first; l < at.layer; l++) {
            if (z < c->layer_zlo[l] || z > c->layer_zhi[l]) continue;
            const int e = executed_in(cts, c->layer_end[l], c, c->layer_jump0[l], c->layer_jump0[l + 1]);
            k += e < 0 ? 0 : e;
        }
    }
    return k;
}
// The growth table as growth.hpp takes it: increments (a step across a binade's boundary reads one)
// and the sums of their deltas, whose first rows a kernel that looks at many cells holds in LDS.
// The chain of a cell's lane is a few reads whatever the number of steps; rounding them one
// after another, up to 63 to catch up and 63 to find the next step due, was the longest part
// of a step of a small domain (50^3 of the finest time step: 23 -> 16 us a step).
struct Growth {
    const double *tab;
    const uint32_t *sums;
    const __attribute__((address_space(3))) uint32_t *staged;  // in LDS (a generic pointer would be read through flat loads)
    int ksat, nstaged;  // rows staged
    double gsat;
    uint32_t usable;
    __device__ __forceinline__ double inc(int k) const { return k < ksat ? tab[k] : gsat; }
    template <typename F>
    __device__ __forceinline__ void with_row(int r, F &&f) const {
        const int at = r * (ksat + 2);
        if (r < nstaged) f(sum_row_at(staged + at, ksat));
        else f(sum_row_at(sums + at, ksat));
    }
};
__device__ __forceinline__ Growth growth_of(const DomainView &d) {
    return Growth{d.grow, d.grow_sums, nullptr, d.ksat, 0, d.gsat, d.sums_usable};
}
// Copies as many rows of the sums as fit to the workgroup's LDS buffer of N entries. Every thread of the
// workgroup calls it.
template <int BLOCK, int N>
__device__ __forceinline__ void stage_sums(const DomainView &d, Growth &g, uint32_t (&lds)[N]) {
    const int len = d.ksat + 2;
    g.staged = (const __attribute__((address_space(3))) uint32_t *)lds;
    g.nstaged = N / len < kSumRows ? N / len : kSumRows;
    const int n = g.nstaged * len;
    const uint4 *src = reinterpret_cast<const uint4 *>(d.grow_sums);
    uint4 *dst = reinterpret_cast<uint4 *>(lds);
    for (int i = threadIdx.x; i < n / 4; i += BLOCK) dst[i] = src[i];
    for (int i = n / 4 * 4 + threadIdx.x; i < n; i += BLOCK) lds[i] = d.grow_sums[i];
    __syncthreads();
}

// dl after the growth of the steps with index k0+1 .. k1, one float rounding per step exactly as
// the reference stores it.
__device__ __forceinline__ float replay_growth(const Growth &g, float dl, int k0, int k1) {
    return advance_steps(g, dl, k0, k1);
}
// Steps ahead (1 .. kAlarmSlots - 1) at which dl, now at growth index k, first reaches thr; the
// horizon when it does not get there before.
__device__ __forceinline__ uint32_t steps_until(const Growth &g, float dl, int k, float thr) {
    return static_cast<uint32_t>(reach_steps(g, dl, k, thr, static_cast<int>(kAlarmSlots) - 1));
}

// ---- The calendar: cell q is processed at the step of serial s when bit q of slot s mod
// kAlarmSlots is set. ----
__device__ __forceinline__ void set_alarm(const DomainView &d, uint32_t serial, uint32_t q) {
    atomicOr(&d.alarms[(serial % kAlarmSlots) * alarm_stride(d.ncell) + (q >> 5)], 1u << (q & 31));
}

// ---- The workgroups that serve one domain in a launch: b of nb. Every body below works for one
// domain; the plain launches use the grid x dimension, the ensemble launches add one grid row per
// domain slot. A finished domain (device-side termination) keeps its state: its bodies return at
// once. ----

// Events of a step counted per workgroup in LDS. A wave adds its lanes' events at once.
__device__ __forceinline__ void count_event(bool happened, uint32_t *counter) {
    const unsigned long long m = __ballot(happened);
    if (m && (threadIdx.x & 63) == static_cast<uint32_t>(__ffsll(static_cast<long long>(m)) - 1))
        atomicAdd(counter, static_cast<uint32_t>(__popcll(m)));
}
// A workgroup's events over some steps, thread e holding those of kind e: their number and the sum of
// the serials of their steps, from which book_totals forms the per-step sums.
struct Tally {
    unsigned long long n = 0, at = 0;
    __device__ __forceinline__ void add(const uint32_t *cnt, uint32_t serial) {
        if (threadIdx.x >= kStepCounts) return;
        const uint32_t c = cnt[threadIdx.x];
        n += c;
        at += static_cast<unsigned long long>(c) * serial;
    }
    // to workgroup b's running totals
    __device__ __forceinline__ void put(const DomainView &d, uint32_t b) {
        if (threadIdx.x >= kStepCounts || !n) return;
        // (an atomic, though nothing else writes the line: it need not wait for the old value)
        unsigned long long *p = d.part + static_cast<size_t>(b) * kPartRows + 2 * threadIdx.x;
        atomicAdd(p, n);
        atomicAdd(p + 1, at);
        n = at = 0;
    }
};
__device__ __forceinline__ void add_parts(const DomainView &d, uint32_t b, const uint32_t *cnt, uint32_t serial) {
    Tally t;
    t.add(cnt, serial);
    t.put(d, b);
}

// Growth index that an active cell's dl includes, at a step of growth index k. A cell not yet
// looked at as an active cell (mask not yet known, or built by its capture: kFresh) holds its
// initial dl: it grows from the step it is first looked at on, so its base is k - 1 (k while it
// waits for its liquidus time or its layer: k then holds only earlier layers' steps, 0 in a
// single-layer run); otherwise the base is in win.
__device__ __forceinline__ int growth_base(const CellWords &w, int k, bool waiting) {
    if ((w.lm & kLmUnknown) || (w.flags & kFresh)) return waiting ? k : k - 1;
    return static_cast<int>(w.win);
}
// Cell r of known mask is past its liquidus time and has no liquid neighbour left: at its visit
// in the capture of the step of growth index k the reference grows it and turns it solid
// (src/CAupdate.cpp:722-725).
__device__ __forceinline__ void solidify(const DomainView &d, const Growth &g, uint32_t r, const CellWords &w, int k) {
    Cell &c = d.cells[r];
    c.dl = replay_growth(g, w.dl, growth_base(w, k, false), k);
    c.win = static_cast<uint32_t>(k);
    c.flags = w.flags & ~kFresh;
    c.ct = kSolid;
}

// Nucleation (src/CAupdate.cpp:67-200). A nucleus leaves the liquid masks of its neighbours; a
// neighbour whose mask this empties and that is past its liquidus time finds no liquid neighbour in
// this step's capture and turns solid here.
// The sites of the layer lie in ascending order of time, so the ones due are the next few from
// `from` on; returns how many sites were decided (a cell that is not liquid never turns liquid
// again, so a site past its time is not looked at after). The new active cells are due in this
// step's capture.
template <int BLOCK>
__device__ __forceinline__ int nucleate_body(const DomainView &d, int cycle, uint32_t serial, int layer, int from,
                                             uint32_t b, uint32_t nb, uint32_t *cnt, uint32_t *lohi) {
    const int i0 = from + static_cast<int>(threadIdx.x);
    int m = __syncthreads_count(i0 < d.nnuclei && d.ntime[i0] <= cycle);
    if (m == BLOCK) {  // more than a round of sites: the end of the run of due ones by bisection
        int lo = from + BLOCK - 1, hi = d.nnuclei;  // ntime[lo] <= cycle < ntime[hi]
        while (hi - lo > 1) {
            const int mid = lo + (hi - lo) / 2;
            if (d.ntime[mid] <= cycle)
                lo = mid;
            else
                hi = mid;
        }
        m = hi - from;
    }
    const Grid gr = grid_of(d);
    for (int k0 = static_cast<int>(b) * 64; k0 < m; k0 += static_cast<int>(nb) * BLOCK) {
        // a wave of consecutive sites per workgroup and turn: few sites are due at once
        const int turn = static_cast<int>(threadIdx.x >> 6) * static_cast<int>(nb) * 64;
        const int k = k0 + turn + static_cast<int>(threadIdx.x & 63);
        bool act = false, inner = false;
        uint32_t nent = 0, nsol = 0;
        if (k < m) {
            const uint32_t q = static_cast<uint32_t>(d.nloc[from + k]);
            const uint32_t tail = reinterpret_cast<const uint32_t *>(d.cells + q)[7];  // lid | ct << 8 | flags
            if (static_cast<int8_t>(tail & 0xFFu) <= layer && ((tail >> 8) & 0xFFu) == kLiquid) {
                const Coord c = decode(q, gr);
                act = true;
                inner = c.x > 0 && c.x < d.X - 1 && c.y > 0 && c.y < d.Y - 1;
                Cell &cq = d.cells[q];
                cq.dl = 0.01f;
                cq.thr = 0.0f;
                cq.lm = kLmUnknown;
                cq.flags = 0;
                cq.ct = kActive | kSeedBit;
                set_centre(d, q, (c.x + d.xoff) + 0.5, (c.y + d.yoff) + 0.5, c.z + 0.5);
                uint32_t valid = valid_neighbours(c, gr.X, gr.Y, gr.nzA);
                const Rows rows = rows_of(d, gr, q, valid);
                // all updates in flight together, then the results
                uint32_t old[26];
#pragma unroll
                for (int l = 0; l < 26; l++)
                    old[l] = ((valid >> l) & 1u) ? atomicAnd(rows.low(l), ~(1u << kOpposite.v[l])) : 0u;
                uint32_t emptied = 0;
#pragma unroll
                for (int l = 0; l < 26; l++)
                    emptied |= static_cast<uint32_t>(((valid >> l) & 1u) &&
                                                     (old[l] & (kMaskUnknown | kMaskNow)) == (1u << kOpposite.v[l])) << l;
                for (uint32_t e = emptied; e; e &= e - 1) {
                    const uint32_t r = q + gr.offset(__builtin_ctz(e));
                    const CellWords w = load_cell(d.cells + r);
                    if ((w.ct & kTypeMask) != kActive || !(cycle > w.cts && w.lid <= layer)) continue;
                    if (!(w.flags & kCounted)) nent++;
                    solidify(d, growth_of(d), r, w, growth_index(d, layer_at(d), w.cts, w.lid, r, cycle));
                    d.cells[r].flags = (w.flags & ~kFresh) | kCounted;
                    nsol++;
                }
                atomicMin(&lohi[0], q);
                atomicMax(&lohi[1], q);
                set_alarm(d, serial, q);
            }
        }
        count_event(act, &cnt[kCntAct]);
        count_event(inner, &cnt[kCntNn]);
        if (nent) atomicAdd(&cnt[kCntEnt], nent);
        if (nsol) atomicAdd(&cnt[kCntSol], nsol);
    }
    return m;
}

// An active cell without a grain: the domain ends with this step (broken: in LDS, or null).
__device__ __forceinline__ void raise(const DomainView &d, uint32_t *broken) {
    atomicOr(&d.ctl->error, 2);
    if (broken) *broken = 1;
}

// Critical lengths of the liquid neighbours of frontier cell j (half-diagonal dlj): claims on
// those reached. thr becomes the least length of the others (the caller stores it), hint the
// record's note of which neighbour that is and of the next-least length (threshold_hint), and
// the claimed mask is returned. The 26 lengths are one aligned 128-byte row: the cell's own
// (stored by its capture) or, for a cell-centred octahedron, its orientation's row of the seed
// table. They are compared all at once and the claims issued after, so a lane's work does not
// depend on its liquid count.
__device__ uint32_t evaluate_claims(const DomainView &d, const Grid &gr, uint32_t j, float dlj, uint32_t liquid,
                                    int32_t gid, uint8_t ct, float &thr, uint16_t &hint, uint32_t *broken) {
    const float *row = d.octa[j].cdl;
    if (ct & kSeedBit) {
        int o = orientation_of(gid);
        if (o < 0) {
            raise(d, broken);
            o = 0;
        }
        row = d.seed_cdl + static_cast<size_t>(kCdlStride) * o;
    }
    float cdl[26];
    const float4 *r4 = reinterpret_cast<const float4 *>(row);
#pragma unroll
    for (int i = 0; i < 6; i++) {
        const float4 v = r4[i];
        cdl[4 * i] = v.x;
        cdl[4 * i + 1] = v.y;
        cdl[4 * i + 2] = v.z;
        cdl[4 * i + 3] = v.w;
    }
    const float2 v2 = reinterpret_cast<const float2 *>(row)[12];
    cdl[24] = v2.x;
    cdl[25] = v2.y;
    // In integer and min/max operations on the lengths, a neighbour that is not liquid (or, for the
    // threshold, reached) counting as infinitely far: conditions of 26 neighbours at once would need
    // more scalar registers than there are. So does one whose length is NaN (of an orientation that the
    // file did not give), which no half-diagonal reaches: a length is not negative, and as an integer a NaN of
    // either sign is greater than infinity. dlj - len then has its sign bit set exactly when dlj < len.
    constexpr uint32_t kInf = 0x7F800000u;
    uint32_t beyond = 0;
    float next = __builtin_inff(), next2 = __builtin_inff();
    int at = -1;
#pragma unroll
    for (int l = 0; l < 26; l++) {
        const uint32_t liq = static_cast<uint32_t>(static_cast<int32_t>(liquid << (31 - l)) >> 31);
        const uint32_t len = min(__float_as_uint(cdl[l]) | ~liq, kInf);
        const uint32_t sign = __float_as_uint(dlj - __uint_as_float(len));
        beyond |= (sign >> 31) << l;
        const uint32_t open = static_cast<uint32_t>(static_cast<int32_t>(sign) >> 31);
        const float v = __uint_as_float((len & open) | (kInf & ~open));
        next2 = fminf(next2, fmaxf(next, v));
        at = v < next ? l : at;
        next = fminf(next, v);
        // four neighbours at a time: their masked lengths and conditions all at once would take 20
        // registers more, and a workgroup a CU less
        if (l % 4 == 3) asm volatile("" : "+v"(liquid), "+v"(dlj), "+v"(beyond), "+v"(next), "+v"(next2), "+v"(at));
    }
    const uint32_t claimed = ~beyond & liquid;
    for (uint32_t m = claimed; m; m &= m - 1) atomicMin(claim_word(d, j + gr.offset(__builtin_ctz(m))), j);
    thr = next;
    hint = threshold_hint(at, next, next2);
    return claimed;
}

// ---- The workgroups of a
// domain share the units of the range of active cells in turn, so that the front, wherever it lies,
// is spread over all of them. ----
constexpr uint32_t kUnitsPerLane = 8;  // units whose words a wave holds at once

struct UnitRange {
    uint32_t u0, n;  // first unit, number of units
};
// The units that may hold a due cell: all of a domain small enough for one round of its workgroups,
// else those of the range of active cells.
template <int BLOCK>
__device__ __forceinline__ bool scans_all(const DomainView &d, uint32_t nb) {
    return d.units <= nb * (BLOCK / 64) * kUnitsPerLane;
}
template <int BLOCK>
__device__ __forceinline__ UnitRange unit_range(const DomainView &d, uint32_t nb) {
    if (scans_all<BLOCK>(d, nb)) return UnitRange{0, d.units};
    const uint32_t lo = d.ctl->elo;
    uint32_t hi = d.ctl->ehi;
    if (lo > hi) return UnitRange{0, 0};
    if (hi >= static_cast<uint64_t>(d.ncell)) hi = static_cast<uint32_t>(d.ncell - 1);
    return UnitRange{lo / kUnitCells, hi / kUnitCells - lo / kUnitCells + 1};
}
// Workgroup b's place among the nb: its k-th unit is unit k * nb + its place. Workgroups are
// dispatched round-robin over the 8 XCDs; with enough of them, runs of nb / 8 units go to the
// workgroups of one XCD, so that neighbouring cells mostly share an L2.
__device__ __forceinline__ uint32_t place_of(uint32_t b, uint32_t nb) {
    return nb >= 64 && nb % 8 == 0 ? (b % 8) * (nb / 8) + b / 8 : b;
}
__device__ __forceinline__ uint32_t *calendar_slot(const DomainView &d, uint32_t serial) {
    return d.alarms + (serial % kAlarmSlots) * alarm_stride(d.ncell);
}
// Entries of a workgroup's region of the claim lists: the cells of the most units it can hold. The
// regions lie in the order of the workgroups' units, so that those of workgroups without any come last.
__device__ __forceinline__ uint32_t claim_region(const DomainView &d, uint32_t nb) {
    return (d.units + nb - 1) / nb * kUnitCells;
}

// Calls visit(has, j, record) for every cell due at the step of that serial in workgroup b's units,
// BLOCK cells at a time in a uniform loop (has: the lane has one). The due cells are gathered in LDS
// (`list`, CAP entries) over as many rounds of units as fit and then processed together, so that the
// lanes are full; a round that does not fit is read again for the rest. With CLEAR the bits of a
// finished round are cleared for the slot's next use, 64 steps on. meanwhile() is called, by every
// thread, while the first words are on their way; false: there is nothing to do after all.
template <int BLOCK, uint32_t CAP, bool CLEAR, typename G, typename F>
__device__ __forceinline__ void for_due(const DomainView &d, uint32_t serial, uint32_t b, uint32_t nb, uint32_t *list,
                                        uint32_t *tot, G &&meanwhile, F &&visit) {
    bool first_words = true;
    constexpr uint32_t kWaves = BLOCK / 64;
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const UnitRange r = unit_range<BLOCK>(d, nb);
    uint32_t *bits = calendar_slot(d, serial);
    // this lane's word of its wave's first unit, and the end of the range's words
    const uint32_t first = (r.u0 + wave * nb + place_of(b, nb)) * kUnitWords + lane;
    const uint32_t end = (r.u0 + r.n) * kUnitWords < d.nwords ? (r.u0 + r.n) * kUnitWords : d.nwords;
    uint32_t fill = 0, done = 0;                // entries in the list; cells of the round already listed
    for (uint32_t k0 = 0; k0 * nb < r.n;) {
        uint32_t w[kUnitsPerLane], cnt = 0;
        auto word = [&](uint32_t e) { return first + (k0 + e * kWaves) * nb * kUnitWords; };
        // all loads in flight together (no test around each: a word past the end reads the last one)
        const uint32_t turns = (r.n - k0 * nb + kWaves * nb - 1) / (kWaves * nb);  // that have a unit at all
#pragma unroll
        for (uint32_t e = 0; e < kUnitsPerLane; e++) {
            w[e] = 0;
            if (e < turns) w[e] = bits[word(e) < end ? word(e) : end - 1];
        }
        if (first_words && !meanwhile()) return;
        first_words = false;
#pragma unroll
        for (uint32_t e = 0; e < kUnitsPerLane; e++) {
            w[e] = word(e) < end ? w[e] : 0u;
            cnt += __builtin_popcount(w[e]);
        }
        uint32_t wtot;
        const uint32_t incl = wave_inclusive_scan(cnt, wtot);
        if (lane == 0) tot[wave] = wtot;
        __syncthreads();
        uint32_t before = 0, total = 0;
#pragma unroll
        for (uint32_t q = 0; q < kWaves; q++) {
            const uint32_t v = tot[q];
            before += q < wave ? v : 0u;
            total += v;
        }
        const uint32_t take = total - done < CAP - fill ? total - done : CAP - fill;
        const bool last = done + take == total;
        uint32_t pos = before + incl - cnt - done;  // place among the cells to list now; wraps if listed before
#pragma unroll
        for (uint32_t e = 0; e < kUnitsPerLane; e++) {
            if (e >= turns || !w[e]) continue;
            if (CLEAR && last) bits[word(e)] = 0u;
            for (uint32_t m = w[e]; m; m &= m - 1, pos++)
                if (pos < take) list[fill + pos] = word(e) * 32u + __builtin_ctz(m);
        }
        fill += take;
        done = last ? 0 : done + take;
        if (last) k0 += kWaves * kUnitsPerLane;
        __syncthreads();  // the list is written, tot is read
        if (fill < CAP && k0 * nb < r.n) continue;
        // software pipeline: the next turn's record is loaded while this one's is processed
        uint32_t jn = 0;
        CellWords wn{};
        if (threadIdx.x < fill) {
            jn = list[threadIdx.x];
            wn = load_cell(d.cells + jn);
        }
        for (uint32_t i0 = 0; i0 < fill; i0 += BLOCK) {
            const uint32_t i = i0 + threadIdx.x;
            const uint32_t j = jn;
            const CellWords wc = wn;
            if (i + BLOCK < fill) {
                jn = list[i + BLOCK];
                wn = load_cell(d.cells + jn);
            }
            visit(i < fill, j, wc);
        }
        fill = 0;
        __syncthreads();  // the list is read
    }
}

// A cell found with a known, empty mask at the step after the one that emptied it. The reference
// visits cells in ascending index order with every capture visible at once, so a cell whose liquid
// neighbours all went to lower-indexed claimants has none left at its visit and turns solid in that
// step; a capture by itself or a later cell leaves it active for one more step (src/CAupdate.cpp:
// 333-334, 722-725). Every capture that took a neighbour of it with a claimant of index >= its own
// left the step's tag in its keep word. serial, cycle: the step after the one that emptied it. A cell
// that waited for its liquidus time or its layer then was not visited in that step.
__device__ __forceinline__ bool solid_since_last(const CellWords &w, uint32_t serial, int cycle, int layer) {
    return !(w.lm & (kLmUnknown | kLmNow)) && !(w.flags & kFresh) && static_cast<uint32_t>(w.lm >> 32) != serial &&
           cycle - 1 > w.cts && w.lid <= layer;
}

// The liquid ones among the 26 neighbours of active cell j, from their types: a plane of nine at a time
// (only a nucleus or a seed asks, once, and 26 reads in flight would cost the claim pass registers).
__device__ __forceinline__ uint32_t liquid_neighbours(const DomainView &d, const Grid &gr, uint32_t j) {
    uint32_t raw = 0;  // bit 9 (dz + 1) + 3 (dx + 1) + dy + 1
#pragma unroll 1
    for (int z = 0; z < 3; z++) {
        const Cell *row = d.cells + static_cast<uint32_t>(j + (z - 1) * static_cast<int>(gr.xy.d));
        uint32_t nine = 0;
#pragma unroll
        for (int i = 0; i < 9; i++)
            nine |= static_cast<uint32_t>(row[(i / 3 - 1) * gr.Y + i % 3 - 1].ct == kLiquid) << i;
        raw |= nine << (9 * z);
    }
    uint32_t liquid = 0;
#pragma unroll
    for (int l = 0; l < 26; l++) liquid |= ((raw >> (9 * (kNbZ[l] + 1) + 3 * (kNbX[l] + 1) + kNbY[l] + 1)) & 1u) << l;
    return liquid;
}

// Pass A over the cells due this step (the step's calendar slot), one per lane: the liquidus-time
// gate, the growth since the cell was last looked at, and the claims.
// The liquid neighbours come from the cell's mask (lm), kept current by the cells that leave the
// liquid state; a new active cell builds it once from the 26 neighbour types. A cell past its
// liquidus time with no liquid neighbour turns solid here (no capture of this step can give it
// one); one that the step before left without any, and that the reference turned solid in that
// step, gets the state of that step (with follows: the step before ran just before, and its
// solidifications are not yet settled).
// thr is a lower bound on the critical length of every neighbour that is still liquid: the
// smallest critical length over the liquid neighbours the cell did not claim when it last
// evaluated them. Liquid sets only shrink and a cell's octahedron centre is
// fixed, so no capture is possible before the half-diagonal reaches thr: the cell is scheduled for
// that step (or for the end of its wait for the liquidus time) and not looked at before, unless a
// neighbour's capture or nucleation empties its mask. A new active cell starts at thr = 0.
// Cells with claims are numbered by an LDS counter (no global atomics) and handed to put(number, cell,
// claimed neighbours).
template <int BLOCK, uint32_t CAP, typename G, typename F>
__device__ __forceinline__ void claim_body(const DomainView &d, const Grid &gr, const Growth &g, const LayerAt &at,
                                           int cycle, uint32_t serial, bool follows, uint32_t b, uint32_t nb,
                                           uint32_t *list, uint32_t *tot, uint32_t *cnt, uint32_t *nclaim,
                                           uint32_t *broken, G &&meanwhile, F &&put) {
    const int layer = at.layer;
    for_due<BLOCK, CAP, true>(d, serial, b, nb, list, tot, meanwhile, [&](bool has, uint32_t j, const CellWords &w) {
        uint32_t claimed = 0;
        bool entered = false, sol = false, late = false, eval = false, mask = false;
        if (has && (w.ct & kTypeMask) == kActive) {
            const bool waiting = !(cycle > w.cts && w.lid <= layer);
            int k = growth_index(d, at, w.cts, w.lid, j, cycle);
            uint32_t liquid;
            const int kdl = growth_base(w, k, waiting);
            // the record's new words, written back as one sector at the end
            unsigned long long lm = w.lm;
            float dl = w.dl, thr = w.thr;
            uint32_t win = w.win;
            uint8_t ct = w.ct;
            uint16_t flags = w.flags;
            if (w.lm & kLmUnknown) {
                const Coord c = decode(j, gr);
                uint32_t valid = valid_neighbours(c, gr.X, gr.Y, gr.nzA);
                liquid = liquid_neighbours(d, gr, inner_cell(d, gr, j, valid)) & valid;
                lm = liquid;
                mask = true;
            }
            else {
                liquid = static_cast<uint32_t>(w.lm & kLmNow);
            }
            if (waiting) {
                win = static_cast<uint32_t>(kdl);
                flags = w.flags & ~kFresh;
                const int ahead = w.cts + 1 - cycle;
                const uint32_t wake = ahead < 1 ? 1u
                                                : (ahead < static_cast<int>(kAlarmSlots) - 1 ? static_cast<uint32_t>(ahead)
                                                                                           : kAlarmSlots - 1);
                set_alarm(d, serial + wake, j);
            }
            else {
                late = follows && solid_since_last(w, serial, cycle, layer);
                if (late) k--;  // the step before: one executed step earlier
                entered = !(w.flags & kCounted);
                flags = (w.flags & ~kFresh) | kCounted;
                dl = replay_growth(g, w.dl, kdl, k);
                win = static_cast<uint32_t>(k);
                if (!liquid) {
                    ct = kSolid;
                    sol = !late;
                }
                else {
                    if (dl >= thr) {
                        const uint32_t set_by = (w.flags >> 2) & 31u;
                        const float bound = hint_bound(thr, w.flags);
                        if (set_by && !((liquid >> (set_by - 1)) & 1u) && dl < bound) {
                            // the neighbour that set thr is gone and no other is reached
                            thr = bound;
                            flags &= ~kHintMask;
                        }
                        else {
                            uint16_t hint = 0;
                            claimed = evaluate_claims(d, gr, j, dl, liquid, w.gid, w.ct, thr, hint, broken);
                            flags = (flags & ~kHintMask) | hint;
                            eval = true;
                        }
                    }
                    // No neighbour left to reach (all claimed now): the captures of this step
                    // empty the mask, and the next step decides the cell's fate.
                    if (thr < __builtin_inff()) set_alarm(d, serial + steps_until(g, dl, k, thr), j);
                }
            }
            // Only this lane writes cell j in this pass (claims go to liquid cells' claim words,
            // mask builds read liquid cells' types), so the whole sector is written back.
            uint4 *r4 = reinterpret_cast<uint4 *>(d.cells + j);
            r4[0] = make_uint4(static_cast<uint32_t>(lm), static_cast<uint32_t>(lm >> 32), __float_as_uint(dl),
                               __float_as_uint(thr));
            r4[1] = make_uint4(static_cast<uint32_t>(w.cts), static_cast<uint32_t>(w.gid), win,
                               static_cast<uint32_t>(static_cast<uint8_t>(w.lid)) | (static_cast<uint32_t>(ct) << 8) |
                                   (static_cast<uint32_t>(flags) << 16));
        }
        const uint32_t slot = wave_append(claimed != 0, nclaim);
        if (claimed) put(slot, j, claimed);
        count_event(entered, &cnt[kCntEnt]);
        count_event(sol, &cnt[kCntSol]);
        count_event(late, &cnt[kCntLate]);
        count_event(eval, &cnt[kCntEval]);
        count_event(mask, &cnt[kCntMask]);
    });
}

// A capture's new octahedron, built by one lane and read by the 32 that give the captured cell its
// place among its neighbours.
struct Capture {
    double cx, cy, cz;
    float gv[9];  // the grain's unit vectors
    float dl;
    uint32_t from, q;  // the winner and the captured cell
    int32_t gid;
};
// LDS of pass B.
template <int BLOCK>
struct ApplyLds {
    // captures to make: the winner, its grain, and the neighbour of it that it captures
    uint32_t from[BLOCK];
    int32_t gid[BLOCK];
    uint8_t which[BLOCK];
    Capture made[BLOCK];
    uint32_t n;
};

// The octahedron of the winner jc's capture of its neighbour l (src/CAupdate.cpp:353-515).
__device__ __forceinline__ void build_capture(const DomainView &d, const Grid &gr, uint32_t jc, int l, int h, Capture &m,
                                              uint32_t *broken) {
    const Octa &e = d.octa[jc];
    // the winner's centre, float as the capture uses it
    const float wcx = static_cast<float>(e.x), wcy = static_cast<float>(e.y), wcz = static_cast<float>(e.z);
    int o = orientation_of(h);
    if (o < 0) {
        raise(d, broken);
        o = 0;
    }
    float gv[9];
#pragma unroll
    for (int i = 0; i < 9; i++) gv[i] = d.guv[9 * o + i];
    const Coord c = decode(jc, gr);
    const double xp = (c.x + d.xoff + nb_dx(l)) + 0.5;
    const double yp = (c.y + d.yoff + nb_dy(l)) + 0.5;
    const double zp = (c.z + nb_dz(l)) + 0.5;
#pragma unroll
    for (int i = 0; i < 9; i++) m.gv[i] = gv[i];
    m.from = jc;
    m.q = jc + gr.offset(l);
    m.gid = h;
    __builtin_amdgcn_sched_barrier(0);  // stored before the octahedron is built: fewer registers live
    const Octahedron oc = new_octahedron(gv, wcx, wcy, wcz, xp, yp, zp);
    m.cx = oc.cx;
    m.cy = oc.cy;
    m.cz = oc.cz;
    m.dl = static_cast<float>(oc.dl);
}

// A lane's neighbour number within its half-wave (26 .. 31: none), its offsets, and the number that the
// cell has as the neighbour's neighbour.
struct NeighbourLane {
    int l, dx, dy, dz, off, back;
};
__device__ __forceinline__ NeighbourLane neighbour_lane(const Grid &gr) {
    NeighbourLane n;
    n.l = static_cast<int>(threadIdx.x & 31u);
    const int l = n.l < 26 ? n.l : 0;
    n.dx = nb_dx(l);
    n.dy = nb_dy(l);
    n.dz = nb_dz(l);
    n.off = gr.offset(l);
    n.back = 0;
#pragma unroll
    for (int i = 0; i < 26; i++) n.back = l == i ? kOpposite.v[i] : n.back;
    return n;
}

// The captured cell's place (src/CAupdate.cpp:553-563, 717), by a half-wave, one lane per neighbour: the
// cell is active, due at the next step and leaves the liquid masks of its neighbours, and its 26
// critical lengths and its centre are written as one line. Only masks that still hold the cell are
// updated: a mask is read first, and a cell's bit is cleared by its capture alone, so the read decides
// exactly. A neighbour whose mask this empties is due at the next step, which decides whether it turned
// solid in this one (solid_since_last). word was read beforehand: the neighbour's lm, and in lanes 26 and
// 27 the last two words of the cell's own record.
__device__ __forceinline__ bool has_neighbour(const DomainView &d, const NeighbourLane &n, const Coord &c) {
    const int x = c.x + n.dx, y = c.y + n.dy, z = c.z + n.dz;
    return n.l < 26 && x >= 0 && x < d.X && y >= 0 && y < d.Y && z >= 0 && z < d.nzA;
}
// A half-wave takes two captures at a time through the three steps (take, write, wake), so that two atomics
// and two sets of next words are in flight: each trip to memory takes 1-2 us at the wide fronts, whose
// cells are far apart. k_apply at 800^3 (cycles 6006-6025, 63 K captures a step) 72 -> 68 us; us a step: 256^3
// 26.0 -> 25.5, 400^3 37.1 -> 36.4, 800x800x40 40.0 -> 39.6, 100^3 14.5 -> 14.3.
struct Placing {
    Coord c;
    unsigned long long word;
    uint32_t liquid, old;
    bool has, valid, need;
};
__device__ __forceinline__ void take_place(const DomainView &d, const NeighbourLane &n, uint32_t serial, const Capture &m,
                                           Placing &a) {
    const uint32_t nb = m.q + n.off, low = static_cast<uint32_t>(a.word), bit = 1u << n.back;
    // The new cell's mask: its liquid neighbours at its first visit are those liquid now and not claimed
    // in this step (every claimed cell is captured in this step, and the claims are final). Until it is
    // stored, the new cell's own words read as a claimed liquid cell, which no other capture counts.
    const unsigned long long ballot = __ballot(a.valid && is_unclaimed_liquid(a.word));
    a.liquid = static_cast<uint32_t>(threadIdx.x & 32u ? ballot >> 32 : ballot);
    a.need = a.valid && (low & (kMaskUnknown | bit)) == bit;
    uint32_t *words = reinterpret_cast<uint32_t *>(&d.cells[nb].lm);
    if (a.need) {
        a.old = atomicAnd(words, ~bit);
        // a neighbour at or below the claimant's index still had q liquid at its visit in the reference's
        // index order: its keep word gets this step's tag (every writer of a step writes the same value)
        if (nb <= m.from) words[1] = serial + 1;
    }
}
__device__ __forceinline__ void write_place(const DomainView &d, const NeighbourLane &n, uint32_t serial, const Capture &m,
                                            const Placing &a) {
    const uint32_t q = m.q;
    const double xp = (a.c.x + d.xoff) + 0.5, yp = (a.c.y + d.yoff) + 0.5, zp = a.c.z + 0.5;
    const float len = critical_length(faces_of(m.gv), xp, yp, zp, m.cx, m.cy, m.cz, n.dx, n.dy, n.dz);
    const uint32_t i = n.l < 26 ? 0u : static_cast<uint32_t>(n.l - 26);
    const double centre = i < 2 ? m.cx : (i < 4 ? m.cy : m.cz);
    const unsigned long long cb = __builtin_bit_cast(unsigned long long, centre);
    const uint32_t half = static_cast<uint32_t>(i & 1u ? cb >> 32 : cb);
    reinterpret_cast<uint32_t *>(&d.octa[q])[n.l] = n.l < 26 ? __float_as_uint(len) : half;
    // The new cell's record, whole: nothing else writes it in this pass.
    if (n.l >= 26 && n.l < 30) {
        unsigned long long w = a.liquid;  // lm (lane 28)
        if (n.l == 26) w = (a.word & 0xFFFFFFFFull) | static_cast<unsigned long long>(static_cast<uint32_t>(m.gid)) << 32;  // cts, gid
        if (n.l == 27) w = (a.word & 0xFFFFFFFFFFull) | static_cast<unsigned long long>(kActive) << 40 | static_cast<unsigned long long>(kFresh) << 48;  // win, lid, ct, flags
        if (n.l == 29) w = __float_as_uint(m.dl);  // dl, thr
        reinterpret_cast<unsigned long long *>(d.cells + q)[n.l < 28 ? n.l - 24 : n.l - 28] = w;
    }
    if (n.l == 30) set_alarm(d, serial + 1, q);
}
__device__ __forceinline__ void wake_emptied(const DomainView &d, const NeighbourLane &n, uint32_t serial, const Capture &m,
                                             const Placing &a) {
    const uint32_t bit = 1u << n.back;
    if (a.need && (a.old & (kMaskUnknown | kMaskNow)) == bit) set_alarm(d, serial + 1, m.q + n.off);
}

// The range of active cells widened by a workgroup's new ones: those of nucleation in lohi (LDS) and
// the captures' least and greatest index per thread. Every thread calls it. The range rarely grows: most
// workgroups need no atomic (elo, ehi: it as it was).
struct NewCells {
    uint32_t lo = 0xFFFFFFFFu, hi = 0;
};
__device__ __forceinline__ void widen_range(const DomainView &d, uint32_t *lohi, const NewCells &n, uint32_t elo,
                                            uint32_t ehi) {
    const uint32_t lo = ~wave_max(~n.lo), hi = wave_max(n.hi);  // in lane 63
    if ((threadIdx.x & 63) == 63 && lo <= hi) {
        atomicMin(&lohi[0], lo);
        atomicMax(&lohi[1], hi);
    }
    __syncthreads();
    if (threadIdx.x == 0 && lohi[0] <= lohi[1]) {
        if (lohi[0] < elo) atomicMin(&d.ctl->elo, lohi[0]);
        if (lohi[1] > ehi) atomicMax(&d.ctl->ehi, lohi[1]);
    }
}
__device__ __forceinline__ void widen_range(const DomainView &d, uint32_t *lohi, const NewCells &n = NewCells{}) {
    widen_range(d, lohi, n, d.ctl->elo, d.ctl->ehi);
}

// Pass B over the claimants that claimant(k, cell, bits) gives. A claim whose word holds the claimant's
// own index is won (the lowest index that reached the cell). The captures won are gathered in LDS over
// as many rounds as fit. A capture's octahedron is built by one lane; its neighbours are then visited by the 26
// lanes of a half-wave, so that the words of three consecutive neighbours are read together, its
// lengths are one store of one line, and its chain is one length and one mask long instead of 26.
// One lane per capture took 242 registers (two waves a SIMD) and about 10 000 cycles for one
// capture, this 121 registers and half the cycles (24^3 9.3 -> 7.4 us a step); at 800^3, 63 000 captures a
// step, the pass takes 72 us against 83 us.
template <int BLOCK, typename F>
__device__ __forceinline__ void apply_body(const DomainView &d, const Grid &gr, uint32_t serial, uint32_t nclaimants,
                                           F &&claimant, ApplyLds<BLOCK> &s, uint32_t *cnt, NewCells &made, uint32_t *broken) {
    const uint32_t lane = threadIdx.x & 63;
    const NeighbourLane n = neighbour_lane(gr);
    if (threadIdx.x == 0) s.n = 0;
    __syncthreads();
    for (uint32_t k0 = 0; k0 < nclaimants; k0 += BLOCK) {
        const uint32_t k = k0 + threadIdx.x;
        uint32_t j = 0, cb = 0, won = 0;
        int32_t gid = 0;
        if (k < nclaimants) {
            claimant(k, j, cb);
            gid = d.cells[j].gid;
            // a claimant mostly has one or two claims: four words in flight at a time
            for (uint32_t m = cb; m;) {
                uint32_t bit[4], cw[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    bit[e] = m & (0u - m);
                    m &= m - 1;
                    cw[e] = *claim_word(d, bit[e] ? j + gr.offset(__builtin_ctz(bit[e])) : j);
                }
#pragma unroll
                for (int e = 0; e < 4; e++) won |= cw[e] == j ? bit[e] : 0u;
            }
        }
        // the captures won go to the list; those that no longer fit wait until it is empty again
        for (bool all = false; !all;) {
            uint32_t wtot, base = 0;
            const uint32_t c = __builtin_popcount(won), incl = wave_inclusive_scan(c, wtot);
            if (lane == 63 && wtot) base = atomicAdd(&s.n, wtot);
            uint32_t pos = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(base), 63)) + incl - c;
            for (; won && pos < BLOCK; won &= won - 1, pos++) {
                s.from[pos] = j;
                s.gid[pos] = gid;
                s.which[pos] = static_cast<uint8_t>(__builtin_ctz(won));
            }
            __syncthreads();
            const uint32_t total = s.n;
            all = total <= BLOCK;
            const uint32_t turn = all ? total : BLOCK;
            __syncthreads();
            if (all && k0 + BLOCK < nclaimants) continue;  // with the next round's
            // the neighbours' words of a half-wave's first capture are on their way while the octahedra
            // are built, and those of its next one while it places one
            constexpr uint32_t kHalves = BLOCK / 32;
            uint32_t i = threadIdx.x >> 5;
            Placing next[2];
            auto fetch = [&]() {
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    const uint32_t iu = i + u * kHalves;
                    next[u].has = iu < turn;
                    next[u].valid = false;
                    if (iu >= turn) continue;
                    const uint32_t q = s.from[iu] + gr.offset(static_cast<int>(s.which[iu]));
                    next[u].c = decode(q, gr);
                    next[u].valid = has_neighbour(d, n, next[u].c);
                    const unsigned long long *p = &d.cells[n.l < 26 ? q + n.off : q].lm + (n.l < 26 ? 0 : n.l - 24);
                    if (next[u].valid || n.l == 26 || n.l == 27) next[u].word = *p;
                }
            };
            fetch();
            if (threadIdx.x < turn)
                build_capture(d, gr, s.from[threadIdx.x], static_cast<int>(s.which[threadIdx.x]), s.gid[threadIdx.x],
                              s.made[threadIdx.x], broken);
            if (threadIdx.x == 0) {
                cnt[kCntCap] += turn;
                s.n = 0;
            }
            __syncthreads();
            while (i < turn) {
                Placing now[2] = {next[0], next[1]};
                const Capture &m0 = s.made[i], &m1 = s.made[now[1].has ? i + kHalves : i];
                made.lo = m0.q < made.lo ? m0.q : made.lo;
                made.hi = m0.q > made.hi ? m0.q : made.hi;
                made.lo = m1.q < made.lo ? m1.q : made.lo;
                made.hi = m1.q > made.hi ? m1.q : made.hi;
                take_place(d, n, serial, m0, now[0]);
                if (now[1].has) take_place(d, n, serial, m1, now[1]);
                i += 2 * kHalves;
                fetch();
                write_place(d, n, serial, m0, now[0]);
                if (now[1].has) write_place(d, n, serial, m1, now[1]);
                wake_emptied(d, n, serial, m0, now[0]);
                if (now[1].has) wake_emptied(d, n, serial, m1, now[1]);
            }
            __syncthreads();
        }
    }
}

// The solidifications that the last executed step left to the next one (solid_since_last), made now
// that a caller looks at the state. The cells are due at the next step, whose calendar slot stays
// as it is. due: the cells due at the next step.
template <int BLOCK, uint32_t CAP>
__device__ __forceinline__ void settle_body(const DomainView &d, const Growth &g, const LayerAt &at, int next_cycle,
                                            uint32_t next_serial, uint32_t b, uint32_t nb, uint32_t *list, uint32_t *tot,
                                            uint32_t *cnt) {
    for_due<BLOCK, CAP, false>(d, next_serial, b, nb, list, tot, [] { return true; }, [&](bool has, uint32_t j, const CellWords &w) {
        const bool late = has && (w.ct & kTypeMask) == kActive && solid_since_last(w, next_serial, next_cycle, at.layer);
        if (late) solidify(d, g, j, w, growth_index(d, at, w.cts, w.lid, j, next_cycle - 1));
        count_event(late, &cnt[kCntLate]);
    });
}

// The running totals since the last booking, summed by one workgroup over the rows of every
// workgroup and added to the run's statistics; the rows start at zero again. With S0 .. S - 1 the
// serials of the steps since then, an event of serial s that adds a cell to a step's count from the
// same step on adds it to S - s steps, one that does so from the step after to S - 1 - s. The
// reference's numSteer of a step: active cells past their liquidus time at the start of its capture
// pass.
template <int BLOCK>
__device__ __forceinline__ void book_totals(const DomainView &d, uint32_t serial_now, unsigned long long *red) {
    StepCtl *ctl = d.ctl;
    // a workgroup's line is read by 16 lanes
    static_assert(kPartRows == 16, "a line of 16 counters per workgroup");
    unsigned long long v0 = 0;
    for (uint32_t i = threadIdx.x; i < d.nparts * kPartRows; i += BLOCK) {
        const unsigned long long x = d.part[i];
        v0 += x;
        if (x) d.part[i] = 0;
    }
    v0 += __shfl_down(v0, 32, 64);
    v0 += __shfl_down(v0, 16, 64);
    if ((threadIdx.x & 63) < kPartRows) red[(threadIdx.x >> 6) * kPartRows + (threadIdx.x & 63)] = v0;
    __syncthreads();
    if (threadIdx.x < kPartRows)
        for (int w = 1; w < BLOCK / 64; w++) red[threadIdx.x] += red[w * kPartRows + threadIdx.x];
    __syncthreads();
    if (threadIdx.x != 0) return;
    const unsigned long long S = serial_now, n = S - ctl->serial_booked;
    const unsigned long long *v = red;
    auto count = [&](int e) { return v[2 * e]; };
    // an event counted in the step of its serial and all later ones, and one from the step after on
    auto from_same = [&](int e) { return S * v[2 * e] - v[2 * e + 1]; };
    auto from_next = [&](int e) { return (S - 1) * v[2 * e] - v[2 * e + 1]; };
    // a late solidification belongs to the step before the one that found it
    const unsigned long long sols = count(kCntSol) + count(kCntLate), sol = from_next(kCntSol) + from_same(kCntLate);
    const unsigned long long frontier = n * ctl->nonwaiting + from_same(kCntEnt) - sol;
    StepStats st = *d.stats;
    st.frontier += frontier;
    st.waiting += n * ctl->nactive + from_same(kCntAct) + from_next(kCntCap) - sol - frontier;
    st.solidified += sols;
    st.captures += count(kCntCap);
    st.activated += count(kCntAct);
    st.nucleated += count(kCntNn);
    st.evaluated += count(kCntEval);
    st.masks += count(kCntMask);
    *d.stats = st;
    ctl->nonwaiting += count(kCntEnt) - sols;
    ctl->nactive += count(kCntAct) + count(kCntCap) - sols;
    ctl->serial_booked = serial_now;
}

// The end of a domain: stopped by an error flag, at the end of the step that raised it (its later steps would
// work on a broken state; the host learns of it at its next check or poll), or, with autostop, at a check step (cycle a
// multiple of 1000) with no liquid left: liquid cells only ever leave the liquid state by capture
// or nucleation, so the reference's superheated + undercooled count (src/CAupdate.cpp:738-783) is
// the initial liquid count minus both.
__device__ __forceinline__ void stop_domain(const DomainView &d, int cycle, int32_t err) {
    d.ctl->done = 1;
    d.ctl->final_cycle = cycle;
    if (err && d.status_err) *d.status_err = err;
    if (d.status) *d.status = cycle;
}
__device__ __forceinline__ void end_domain(const DomainView &d, int cycle) {
    StepCtl *ctl = d.ctl;
    const int32_t err = ctl->error;
    const bool finished = d.autostop && cycle % 1000 == 0 &&
                          d.liquid0 - static_cast<long long>(d.stats->captures) -
                                  static_cast<long long>(d.stats->activated) == 0;
    if (err || finished) stop_domain(d, cycle, err);
}

// Every active cell of the window due at the next step (after a cycle jump, whose skipped steps the
// calendar did not count). Active cells above the window (substrate cells next to a later layer's
// melt pool) are never stepped, as the reference's pass 1 never visits them.
__global__ __launch_bounds__(kBlock) void k_rewake(DomainView d, int p_next) {
    const StepCtl *ctl = d.ctl;
    const uint32_t lo = ctl->elo, hi = ctl->ehi;
    if (lo > hi) return;
    const unsigned long long end = static_cast<unsigned long long>(d.X) * d.Y * d.nzA;
    const uint32_t serial = ctl->serial[p_next];
    for (unsigned long long q = lo + static_cast<unsigned long long>(blockIdx.x) * kBlock + threadIdx.x; q <= hi && q < end;
         q += static_cast<unsigned long long>(gridDim.x) * kBlock)
        if ((d.cells[q].ct & kTypeMask) == kActive) set_alarm(d, serial, static_cast<uint32_t>(q));
}

// The next layer's window (src/CAinitialize.cpp:2772-2832): the plane of the lowest active cell and
// the top plane of the next layer's cells. out[0] = least z (atomicMin), out[1] = greatest z.
__global__ __launch_bounds__(kBlock) void k_layer_bounds(DomainView d, int next_layer, int *out) {
    int zmin = 0x7FFFFFFF, zmax = -1;
    const Grid gr = grid_of(d);
    for (long long q = static_cast<long long>(blockIdx.x) * kBlock + threadIdx.x; q < d.ncell;
         q += static_cast<long long>(gridDim.x) * kBlock) {
        const uint32_t tail = reinterpret_cast<const uint32_t *>(d.cells + q)[7];
        const int z = static_cast<int>(gr.xy.div(static_cast<uint32_t>(q)));
        if (((tail >> 8) & kTypeMask) == kActive) zmin = z < zmin ? z : zmin;
        if (static_cast<int8_t>(tail & 0xFFu) == next_layer) zmax = z > zmax ? z : zmax;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const int a = __shfl_xor(zmin, o, 64), b = __shfl_xor(zmax, o, 64);
        zmin = a < zmin ? a : zmin;
        zmax = b > zmax ? b : zmax;
    }
    if ((threadIdx.x & 63) == 0) {
        atomicMin(&out[0], zmin);
        atomicMax(&out[1], zmax);
    }
}

// LayerSetup (src/CAinitialize.cpp:2835-2982) on the resident state: every active cell of the new
// window [zlo, nzA) gets a cell-centred octahedron (half-diagonal 0.01, centre at the cell centre,
// critical lengths from its orientation) and an unknown liquid mask (its neighbours changed with the
// layer), is counted afresh, and is due at the first step of the layer (the step of parity p_next).
// The calendar was cleared before. ctl->nactive and the range of active
// cells (ctl->elo, ctl->ehi, reset by the host) are accumulated here.
__global__ __launch_bounds__(kBlock) void k_layer_setup(DomainView d, int p_next) {
    __shared__ unsigned long long sh[kBlock / 64];
    StepCtl *ctl = d.ctl;
    const uint32_t serial = ctl->serial[p_next];
    const Grid gr = grid_of(d);
    const long long begin = static_cast<long long>(d.X) * d.Y * d.zlo;
    const long long end = static_cast<long long>(d.X) * d.Y * d.nzA;
    unsigned long long n = 0;
    uint32_t qlo = 0xFFFFFFFFu, qhi = 0;
    for (long long q = begin + static_cast<long long>(blockIdx.x) * kBlock + threadIdx.x; q < end;
         q += static_cast<long long>(gridDim.x) * kBlock) {
        Cell &c = d.cells[q];
        if ((c.ct & kTypeMask) != kActive) continue;
        const Coord p = decode(static_cast<uint32_t>(q), gr);
        c.lm = kLmUnknown;
        c.dl = 0.01f;
        c.thr = 0.0f;
        c.win = 0;
        c.flags = 0;
        c.ct = kActive | kSeedBit;
        set_centre(d, q, (p.x + d.xoff) + 0.5, (p.y + d.yoff) + 0.5, p.z + 0.5);
        set_alarm(d, serial, static_cast<uint32_t>(q));
        n++;
        qlo = static_cast<uint32_t>(q) < qlo ? static_cast<uint32_t>(q) : qlo;
        qhi = static_cast<uint32_t>(q) > qhi ? static_cast<uint32_t>(q) : qhi;
    }
    const unsigned long long t = block_sum(n, sh);
    if (threadIdx.x == 0 && t) atomicAdd(&ctl->nactive, t);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const uint32_t a = __shfl_xor(qlo, o, 64), b = __shfl_xor(qhi, o, 64);
        qlo = a < qlo ? a : qlo;
        qhi = b > qhi ? b : qhi;
    }
    if ((threadIdx.x & 63) == 0 && qlo <= qhi) {
        atomicMin(&ctl->elo, qlo);
        atomicMax(&ctl->ehi, qhi);
    }
}

// LDS of a workgroup's step counters and of the range of its new active cells.
struct StepTally {
    uint32_t cnt[kStepCounts];
    uint32_t lohi[2];
};
__device__ __forceinline__ void clear_tally(StepTally &t) {
    if (threadIdx.x < kStepCounts) t.cnt[threadIdx.x] = 0;
    if (threadIdx.x < 2) t.lohi[threadIdx.x] = threadIdx.x == 0 ? 0xFFFFFFFFu : 0u;
    __syncthreads();
}
// Whether the step at `cycle` directly follows the last executed one (no cycle jump, same layer).
__device__ __forceinline__ bool follows_last(const StepCtl *ctl, int cycle) {
    return cycle > 1 && ctl->last_cycle == cycle - 1;
}
constexpr uint32_t kDueStage = 1024;  // due cells of a turn staged in LDS
constexpr int kClaimSums = 8192;      // entries of the growth sums staged in LDS by every claim workgroup

// A step's kernels get its cycle and serial as arguments: a kernel's first loads find cold caches, and each
// one that others wait for costs 1.5 us of every step. What else they need first is asked for together:
// the claim pass reads its calendar words while it stages the growth sums (all the rows of a
// coarse time step: a row read from memory costs the cells on it that time for every probe), the apply pass its
// claimants before it knows how many there are. us a step without and with: 256^3 29.7, 26.0; 400^3 41.5,
// 37.1; 800^3 (cycles 6006-6025) 161, 155.
__device__ __forceinline__ void nucleate_step(const DomainView &d, int cycle, uint32_t serial, uint32_t b, uint32_t nb) {
    __shared__ StepTally t;
    StepCtl *ctl = d.ctl;
    if (ctl->done | ctl->halted) return;
    const int from = ctl->nuc_at;
    clear_tally(t);
    const int m = nucleate_body<kBlock>(d, cycle, serial, d.layer, from, b, nb, t.cnt, t.lohi);
    if (b == 0 && threadIdx.x == 0) ctl->nuc_next = from + m;
    if (!m) return;
    widen_range(d, t.lohi);
    add_parts(d, b, t.cnt, serial);
}
__device__ __forceinline__ void claim_step(const DomainView &d, int cycle, uint32_t serial, bool follows, uint32_t b,
                                           uint32_t nb) {
    __shared__ StepTally t;
    __shared__ uint32_t nclaim;
    __shared__ __attribute__((aligned(16))) uint32_t gsums[kClaimSums];
    __shared__ uint32_t list[kDueStage], tot[kBlock / 64];
    const int done = d.ctl->done | d.ctl->halted;
    if (threadIdx.x == 0) nclaim = 0;
    clear_tally(t);
    Growth g = growth_of(d);
    const uint32_t region = place_of(b, nb) * claim_region(d, nb);
    claim_body<kBlock, kDueStage>(
        d, grid_of(d), g, layer_at(d), cycle, serial, follows, b, nb, list, tot, t.cnt, &nclaim, nullptr,
        [&] {
            stage_sums<kBlock>(d, g, gsums);
            return !done;
        },
        [&](uint32_t k, uint32_t j, uint32_t claimed) {
            d.claim_cell[region + k] = j;
            d.claim_bits[region + k] = claimed;
        });
    __syncthreads();
    if (threadIdx.x == 0) d.claim_count[b * kCountStride] = nclaim;
    add_parts(d, b, t.cnt, serial);
}
__device__ __forceinline__ void apply_step(const DomainView &d, int cycle, uint32_t serial, int p, uint32_t a, uint32_t nbc) {
    __shared__ StepTally t;
    __shared__ ApplyLds<kBlock> s;
    StepCtl *ctl = d.ctl;
    const uint32_t region = place_of(a, nbc) * claim_region(d, nbc);
    // (a region has room for more claimants than a workgroup has threads; a workgroup without units has
    // neither claimants nor a region)
    const uint32_t early = (place_of(a, nbc) < d.units ? region : 0u) + threadIdx.x;
    const uint32_t n = d.claim_count[a * kCountStride], cell0 = d.claim_cell[early], bits0 = d.claim_bits[early], elo = ctl->elo, ehi = ctl->ehi;
    // (an error of this step's claims, or of an earlier step, after which nothing is claimed; see steps_body)
    const int32_t err = ctl->error, halted = ctl->halted;
    if (ctl->done) return;
    clear_tally(t);
    NewCells made;
    apply_body<kBlock>(
        d, grid_of(d), serial, n,
        [&](uint32_t k, uint32_t &j, uint32_t &bits) {
            j = k < kBlock ? cell0 : d.claim_cell[region + k];
            bits = k < kBlock ? bits0 : d.claim_bits[region + k];
        },
        s, t.cnt, made, nullptr);
    widen_range(d, t.lohi, made, elo, ehi);
    add_parts(d, a, t.cnt, serial);
    if (a == 0 && threadIdx.x == 0 && !halted) {
        // control words for the kernels that read them there
        ctl->last_cycle = cycle;
        ctl->cycle[1 - p] = cycle + 1;
        ctl->serial[1 - p] = serial + 1;
        ctl->nuc_at = max(ctl->nuc_at, ctl->nuc_next);
        if (err) {  // the last step: of whatever parity the host goes on to, it is settled and booked
            ctl->halted = 1;
            ctl->cycle[p] = cycle + 1;
            ctl->serial[p] = serial + 1;
        }
    }
}
__device__ __forceinline__ void settle_step(const DomainView &d, int p_next, uint32_t b, uint32_t nb) {
    __shared__ StepTally t;
    __shared__ uint32_t list[kDueStage], tot[kBlock / 64];
    StepCtl *ctl = d.ctl;
    if (ctl->done || !follows_last(ctl, ctl->cycle[p_next])) return;
    clear_tally(t);
    const uint32_t serial = ctl->serial[p_next];
    settle_body<kBlock, kDueStage>(d, growth_of(d), layer_at(d), ctl->cycle[p_next], serial, b, nb, list, tot, t.cnt);
    __syncthreads();
    add_parts(d, b, t.cnt, serial);
}
__device__ __forceinline__ void book_step(const DomainView &d, int p_next) {
    __shared__ unsigned long long red[kPartRows * (kBlock / 64)];
    if (d.ctl->done) return;
    book_totals<kBlock>(d, d.ctl->serial[p_next], red);
    if (threadIdx.x == 0) end_domain(d, d.ctl->last_cycle);
}

// ---- A team of workgroups that runs many steps of one domain in one launch. ----

// The team's barrier: every workgroup posts the barrier's number in its own word and waits for all
// the others' words (each polls all of them: one hop. With the waits below and a wave's stores to write back
// 1.7, 2.1, 2.6, 4.5 us for 8, 16, 32, 64 workgroups; with none 1.4, 1.7, 1.9, 4.0). What the team wrote before it
// is visible to the team after it (agent-scope release and acquire by one wave, ordered with the rest
// of the workgroup by its own barriers). A team of one needs the workgroup's barrier alone.
// All of the team's workgroups run (they met before), so every wait ends; it is bounded all the same
// (d.barrier_wait): past it the domain is stopped with error 16 at the step that was being taken, and
// false returned to every thread. Nothing else of that launch is undone or completed: the barrier's number,
// the cycle and the serial stay those of the launch's start, and no later launch takes the domain up.
// broken (LDS): whether an error was raised. After a step's claims (claims) every workgroup learns of every
// other's, so that all stop after the same step. A word read there may already be the next barrier's, of the same
// step: its bit was set by that step's claims or by a capture, whose error a claim of the same step raised
// before it. The other barriers don't look: a word read there may be of the next step.
// Waits until this wave's stores and atomics, and its write-back or invalidation of a cache, have been
// done. The compiler leaves such a wait out where it counts nothing outstanding, and it doesn't count a
// write-back: without this one the barrier's word was stored right behind the write-back's start
// (`buffer_wbl2`), and another XCD could see the word while records were still dirty in this one's L2.
__device__ __forceinline__ void drain() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
struct Team {
    uint32_t b, nb;
    uint32_t number;  // of the last barrier passed, twice; bit 0 of a posted word: an error was raised
};
__device__ __forceinline__ bool team_sync(const DomainView &d, Team &t, int cycle, uint32_t &broken,
                                          bool claims = false) {
    if (t.nb == 1) {
        __syncthreads();
        return true;
    }
    drain();  // every wave its own: the release below waits for its wave's alone
    __syncthreads();
    t.number += 2;
    bool late = false;
    if (threadIdx.x < 64) {
        if (threadIdx.x == 0) {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
            drain();
            __hip_atomic_store(d.sync + t.b, t.number | broken, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (threadIdx.x < t.nb) {
            const unsigned long long t0 = wall_clock64();
            uint32_t word;
            while (static_cast<int32_t>((word = __hip_atomic_load(d.sync + threadIdx.x, __ATOMIC_RELAXED,
                                                                  __HIP_MEMORY_SCOPE_AGENT)) -
                                        t.number) < 0) {
                if (wall_clock64() - t0 > d.barrier_wait) {
                    late = true;
                    break;
                }
            }
            if (claims && (word & 1u)) broken = 1;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        drain();  // the other waves' loads follow the invalidation, not just this one's
    }
    if (!__syncthreads_or(late)) return true;
    if (threadIdx.x == 0) stop_domain(d, cycle, atomicOr(&d.ctl->error, 16) | 16);
    return false;
}

// A team's meeting (meet.hpp), by one wave of each workgroup, a lane to a word; every lane calls and gets the
// same. Two trips to memory where all run.
struct MeetWords {
    const DomainView &d;
    uint32_t b, nb;
    unsigned long long launch, t0, seen;  // seen: what this lane's word held
    __device__ __forceinline__ unsigned long long *word(uint32_t i) const {
        return reinterpret_cast<unsigned long long *>(d.sync + kSyncReports) + i;
    }
    __device__ __forceinline__ void report() const {
        if (threadIdx.x == 0)
            (void)__hip_atomic_fetch_max(word(b), static_cast<unsigned long long>(meet_reported(launch)), __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ __forceinline__ Met look() {
        seen = __hip_atomic_load(word(threadIdx.x < nb ? threadIdx.x : b), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return Met{__all(seen == meet_reported(launch)) != 0, __any(seen == meet_refused(launch)) != 0};
    }
    __device__ __forceinline__ bool expired() const {
        return static_cast<unsigned long long>(wall_clock64()) - t0 >= d.meet_wait;
    }
    __device__ __forceinline__ void refuse() const {
        unsigned long long was = seen;
        if (threadIdx.x < nb && seen < meet_reported(launch))
            (void)__hip_atomic_compare_exchange_strong(word(threadIdx.x), &was,
                                                       static_cast<unsigned long long>(meet_refused(launch)),
                                                       __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
};
// Whether this workgroup takes part in the launch; the team is then all of it, or this one alone. role: LDS.
__device__ __forceinline__ bool team_meets(const DomainView &d, Team &t, unsigned long long launch, uint32_t &role) {
    if (t.nb == 1) return true;
    if (threadIdx.x < 64) {
        Meet m = t.b == 0 ? Meet::kAlone : Meet::kLeave;  // (given no time at all)
        if (d.meet_wait) {
            MeetWords w{d, t.b, t.nb, launch, static_cast<unsigned long long>(wall_clock64()), 0};
            m = meet(w, t.b);
        }
        if (threadIdx.x == 0) role = static_cast<uint32_t>(m);
    }
    __syncthreads();
    if (role == static_cast<uint32_t>(Meet::kAlone)) {
        t.nb = 1;
        if (threadIdx.x == 0) d.ctl->alone++;
    }
    return role != static_cast<uint32_t>(Meet::kLeave);
}

constexpr int kTeamSums = 12288;        // entries of the growth sums staged in LDS
constexpr uint32_t kTeamDue = 2048;     // due cells of a turn staged in LDS

struct TeamLds {
    __attribute__((aligned(16))) uint32_t sums[kTeamSums];
    ApplyLds<kTeamBlock> apply;
    uint32_t list[kTeamDue];
    uint32_t claim_cell[kTeamClaims], claim_bits[kTeamClaims];
    uint32_t tot[kTeamBlock / 64];
    uint32_t nclaim, role;
    uint32_t broken;  // an error was raised, here or by the time of the last barrier elsewhere in the team
    StepTally tally[2];
    unsigned long long red[kPartRows * (kTeamBlock / 64)];
};

// nsteps steps of one domain (nucleate: their nucleation too), settled and booked at the end. Two
// barriers a step: the claims of a step before its winners, its captures before the next step's due
// cells; a step with a nucleation site due has one more. Control words and counters stay in registers
// and LDS, the growth table in LDS, and caches and code stay warm from step to step.
__device__ __forceinline__ void steps_body(const DomainView &d, int p, int layer, int nsteps, bool nucleate, uint32_t b,
                                           uint32_t team_size, unsigned long long launch, TeamLds &s) {
    StepCtl *ctl = d.ctl;
    if (ctl->done) return;
    Team team{b, team_size, ctl->barrier};
    if (!team_meets(d, team, launch, s.role)) return;
    const uint32_t nb = team.nb;
    int cycle = ctl->cycle[p];
    uint32_t serial = ctl->serial[p];
    bool follows = follows_last(ctl, cycle);
    int site = max(ctl->nuc_at, ctl->nuc_next);
    int next_site = nucleate && site < d.nnuclei ? d.ntime[site] : 0x7FFFFFFF;
    // a launch of a few steps would not earn back what it stages
    Growth g = growth_of(d);
    if (nsteps >= 8) stage_sums<kTeamBlock>(d, g, s.sums);
    const uint32_t region = place_of(b, nb) * claim_region(d, nb);
    const bool whole = scans_all<kTeamBlock>(d, nb);
    const Grid gr = grid_of(d);
    const LayerAt at = layer_at(d);
    if (threadIdx.x == 0) s.broken = 0;
    clear_tally(s.tally[0]);
    clear_tally(s.tally[1]);
    Tally acc;
    NewCells made;
    const int p_end = (p + nsteps) & 1;
    while (nsteps > 0) {
        // a domain with autostop is looked at after every step whose cycle is a multiple of 1000
        int n = nsteps;
        if (d.autostop && n > 1000 - (cycle - 1) % 1000) n = 1000 - (cycle - 1) % 1000;
        nsteps -= n;
        for (; n > 0; n--) {
            StepTally &t = s.tally[serial & 1], &before = s.tally[(serial & 1) ^ 1];
            if (cycle >= next_site) {
                site += nucleate_body<kTeamBlock>(d, cycle, serial, layer, site, b, nb, t.cnt, t.lohi);
                next_site = site < d.nnuclei ? d.ntime[site] : 0x7FFFFFFF;
                if (!whole) widen_range(d, t.lohi);
                if (!team_sync(d, team, cycle, s.broken)) return;
            }
            if (threadIdx.x == 0) s.nclaim = 0;
            __syncthreads();
            claim_body<kTeamBlock, kTeamDue>(d, gr, g, at, cycle, serial, follows, b, nb, s.list, s.tot, t.cnt, &s.nclaim,
                                             &s.broken, [] { return true; }, [&](uint32_t k, uint32_t j, uint32_t claimed) {
                                                 if (k < d.claim_stage) {
                                                     s.claim_cell[k] = j;
                                                     s.claim_bits[k] = claimed;
                                                 }
                                                 else {
                                                     if (k == d.claim_stage) atomicAdd(&ctl->spilled, 1u);
                                                     d.claim_cell[region + k] = j;
                                                     d.claim_bits[region + k] = claimed;
                                                 }
                                             });
            if (!team_sync(d, team, cycle, s.broken, true)) return;
            // (0: an error, and the domain stops at the end of this step. Read with the number of claimants, and no
            // branch out of the loop: with one, 24^3 cells take 6.98 us a step instead of 6.84)
            const int go = 1 - __builtin_amdgcn_readfirstlane(static_cast<int>(s.broken));
            if (threadIdx.x < kStepCounts) before.cnt[threadIdx.x] = 0;
            apply_body<kTeamBlock>(
                d, gr, serial, s.nclaim,
                [&](uint32_t k, uint32_t &j, uint32_t &bits) {
                    j = k < d.claim_stage ? s.claim_cell[k] : d.claim_cell[region + k];
                    bits = k < d.claim_stage ? s.claim_bits[k] : d.claim_bits[region + k];
                },
                s.apply, t.cnt, made, &s.broken);
            if (!whole) widen_range(d, t.lohi, made);
            if (!team_sync(d, team, cycle, s.broken)) return;
            acc.add(t.cnt, serial);
            follows = true;
            cycle++;
            serial++;
            n *= go;
        }
        if (s.broken) nsteps = 0;
        StepTally &t = s.tally[serial & 1], &before = s.tally[(serial & 1) ^ 1];
        settle_body<kTeamBlock, kTeamDue>(d, g, at, cycle, serial, b, nb, s.list, s.tot, t.cnt);
        widen_range(d, t.lohi, made);
        widen_range(d, before.lohi);
        acc.add(t.cnt, serial);
        acc.put(d, b);
        if (!team_sync(d, team, cycle, s.broken)) return;
        clear_tally(s.tally[0]);
        clear_tally(s.tally[1]);
        if (b == 0) {
            book_totals<kTeamBlock>(d, serial, s.red);
            if (threadIdx.x == 0) {
                ctl->last_cycle = cycle - 1;
                ctl->nuc_at = site;
                end_domain(d, cycle - 1);
                ctl->cycle[p_end] = cycle;
                ctl->serial[p_end] = serial;
                ctl->barrier = team.number + 2 * (nsteps > 0);  // with the barrier below
            }
        }
        follows = false;  // settled
        if (nsteps > 0) {
            if (!team_sync(d, team, cycle, s.broken)) return;
            if (ctl->done) return;
        }
    }
}

// Plain launches: one domain, passed by value.
__global__ __launch_bounds__(kBlock) void k_nucleate(DomainView d, int cycle, uint32_t serial) {
    nucleate_step(d, cycle, serial, blockIdx.x, gridDim.x);
}
__global__ __launch_bounds__(kBlock) void k_claim(DomainView d, int cycle, uint32_t serial, int follows) {
    claim_step(d, cycle, serial, follows != 0, blockIdx.x, gridDim.x);
}
__global__ __launch_bounds__(kBlock) void k_apply(DomainView d, int cycle, uint32_t serial, int p) {
    apply_step(d, cycle, serial, p, blockIdx.x, gridDim.x);
}
__global__ __launch_bounds__(kBlock) void k_settle(DomainView d, int p_next) {
    settle_step(d, p_next, blockIdx.x, gridDim.x);
}
__global__ __launch_bounds__(kBlock) void k_book(DomainView d, int p_next) { book_step(d, p_next); }
__global__ __launch_bounds__(kTeamBlock) void k_steps(DomainView d, int p, int layer, int nsteps, int nucleate,
                                                      unsigned long long launch) {
    __shared__ TeamLds s;
    steps_body(d, p, layer, nsteps, nucleate != 0, blockIdx.x, gridDim.x, launch, s);
}

// Ensemble launches: workgroup i is workgroup b of the team of nb that serves the domain of one slot
// (its TeamPlace); a team's workgroups follow one another. Views and places lie in tables that no
// kernel writes, read as constants so that a view is kept in scalar registers like an argument.
template <typename T>
__device__ __forceinline__ T load_constant(const T *table, uint32_t i) {
    static_assert(sizeof(T) % 4 == 0, "whole words");
    struct Words {
        uint32_t w[sizeof(T) / 4];
    } v;
    const auto *src = (const __attribute__((address_space(4))) uint32_t *)(table + i);
#pragma unroll
    for (uint32_t k = 0; k < sizeof(T) / 4; k++) v.w[k] = src[k];
    return __builtin_bit_cast(T, v);
}
// A pointer that comes from memory may lie in any address space for the compiler, and an access through such a
// one (flat) waits for the LDS operations too. ms for all solves without and with: 64 domains of sides 32-64
// 243, 236; 256 of 32-64 445, 433; 16 of 64-192 291, 284; 256 of 32-256 3438, 3377.
template <typename T>
__device__ __forceinline__ void to_global(T *&p) {
    p = (T *)(__attribute__((address_space(1))) T *)reinterpret_cast<uintptr_t>(p);
}
__device__ __forceinline__ DomainView load_view(const DomainView *views, uint32_t slot) {
    DomainView d = load_constant(views, slot);
    to_global(d.cells), to_global(d.octa), to_global(d.claim_cell), to_global(d.claim_bits), to_global(d.claim_count);
    to_global(d.nloc), to_global(d.ntime), to_global(d.guv), to_global(d.seed_cdl), to_global(d.grow);
    to_global(d.grow_sums), to_global(d.ctl), to_global(d.stats), to_global(d.part), to_global(d.alarms);
    to_global(d.sync), to_global(d.status), to_global(d.status_err);
    return d;
}
__global__ __launch_bounds__(kTeamBlock) void k_steps_n(const DomainView *views, const TeamPlace *places, int layer,
                                                        int nsteps, unsigned long long launch) {
    __shared__ TeamLds s;
    const TeamPlace at = load_constant(places, blockIdx.x);
    const DomainView d = load_view(views, at.slot);
    steps_body(d, 0, layer, nsteps, true, at.b, at.nb, launch, s);
}

__global__ __launch_bounds__(kBlock) void k_check(DomainView d, int cycle, int layer, CheckResult *out) {
    __shared__ unsigned long long sh[kBlock / 64];
    __shared__ unsigned long long shmin[kBlock / 64];
    unsigned long long c[5] = {0, 0, 0, 0, 0};
    unsigned long long next = ~0ull, amin = ~0ull, amax = 0;
    // the active window [ZBound_Low, ZBound_High] (src/CAupdate.cpp:792-808 reduces over it)
    const long long active_begin = static_cast<long long>(d.X) * d.Y * d.zlo;
    const long long active_end = static_cast<long long>(d.X) * d.Y * d.nzA;
    for (long long q = static_cast<long long>(blockIdx.x) * kBlock + threadIdx.x; q < d.ncell;
         q += static_cast<long long>(gridDim.x) * kBlock) {
        const int t = d.cells[q].ct & kTypeMask;
        if (t == kActive && q >= active_begin && q < active_end) {
            amin = static_cast<unsigned long long>(q) < amin ? static_cast<unsigned long long>(q) : amin;
            amax = static_cast<unsigned long long>(q) > amax ? static_cast<unsigned long long>(q) : amax;
        }
        if (d.cells[q].lid == layer) {
            if (t == kLiquid) {
                const int crit = d.cells[q].cts;
                if (crit > cycle)
                    c[0]++;
                else
                    c[1]++;
                const unsigned long long v = static_cast<unsigned long long>(static_cast<long long>(crit));
                if (q >= active_begin && q < active_end && v < next) next = v;
            }
            else if (t == kActive)
                c[2]++;
            else if (t == kSolid)
                c[3]++;
        }
        else if (t == kLiquid) {
            c[4]++;
        }
    }
    for (int k = 0; k < 5; k++) {
        const unsigned long long s = block_sum(c[k], sh);
        if (threadIdx.x == 0 && s) atomicAdd(&out->counts[k], s);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long v = __shfl_down(next, o, 64);
        next = v < next ? v : next;
    }
    if ((threadIdx.x & 63) == 0) shmin[threadIdx.x >> 6] = next;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long m = shmin[0];
        for (int q = 1; q < kBlock / 64; q++) m = shmin[q] < m ? shmin[q] : m;
        if (m != ~0ull) atomicMin(&out->next_cts, m);
    }
    // range of the active cells, one atomic per wave
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long a = __shfl_down(amin, o, 64), b = __shfl_down(amax, o, 64);
        amin = a < amin ? a : amin;
        amax = b > amax ? b : amax;
    }
    if ((threadIdx.x & 63) == 0 && amin <= amax) {
        atomicMin(&out->amin, amin);
        atomicMax(&out->amax, amax);
    }
}

__global__ __launch_bounds__(kBlock) void k_seed_init(DomainView d, const uint32_t *cells, uint32_t n) {
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        const uint32_t q = cells[i];
        const Coord c = decode(q, d.X, d.Y);
        d.cells[q].dl = 0.01f;
        set_centre(d, q, (c.x + d.xoff) + 0.5, (c.y + d.yoff) + 0.5, c.z + 0.5);
        set_alarm(d, 0, q);
    }
}

// Grain statistics of a region of the whole-domain views (k, i, j), the layout the reference's vtk
// files and its analysis executable use (analysis/src/GAprint.cpp:17-108): the interior of this
// domain for z = 1 .. nz-2, zero on the bottom and top planes. Per cell: its GrainID is flagged in
// gflag (GrainID - gmin; plain stores: every writer writes 1), a negative one counts as nucleated,
// and a melted cell counts in the bin of its orientation (LDS bins flushed once per workgroup), in
// a second set of bins when it lies in the region's top plane.
__global__ __launch_bounds__(kBlock) void k_grain_stats(DomainView d, const uint8_t *melted, GrainRegion r, int gmin,
                                                        uint32_t ngid, uint32_t *gflag, unsigned long long *counts,
                                                        unsigned int *obins, unsigned int *otop) {
    __shared__ unsigned int bins[kNumOrientations];
    __shared__ unsigned long long sh[kBlock / 64];
    for (int o = threadIdx.x; o < kNumOrientations; o += kBlock) bins[o] = 0;
    __syncthreads();
    const long long ni = r.i1 - r.i0 + 1, nj = r.j1 - r.j0 + 1, nk = r.k1 - r.k0 + 1;
    const long long total = ni * nj * nk;
    unsigned long long nmelt = 0, nnuc = 0, nbad = 0;
    for (long long c = static_cast<long long>(blockIdx.x) * kBlock + threadIdx.x; c < total;
         c += static_cast<long long>(gridDim.x) * kBlock) {
        const int j = r.j0 + static_cast<int>(c % nj);
        const int i = r.i0 + static_cast<int>((c / nj) % ni);
        const int k = r.k0 + static_cast<int>(c / (nj * ni));
        int g = 0;
        bool m = false;
        if (k >= 1 && k <= d.nz - 2) {
            const long long q = (static_cast<long long>(k) * d.X + (i + 1)) * d.Y + (j + 1);
            g = d.cells[q].gid;
            m = melted[q] != 0;
        }
        const long long f = static_cast<long long>(g) - gmin;
        if (f < 0 || f >= ngid) {
            nbad++;
            continue;
        }
        gflag[f] = 1u;
        nnuc += g < 0;
        if (m) {
            nmelt++;
            const int o = orientation_of(g) < 0 ? 0 : orientation_of(g);
            atomicAdd(&bins[o], 1u);
            if (k == r.k1) atomicAdd(&otop[o], 1u);
        }
    }
    const unsigned long long tm = block_sum(nmelt, sh);
    const unsigned long long tn = block_sum(nnuc, sh);
    const unsigned long long tb = block_sum(nbad, sh);
    if (threadIdx.x == 0) {
        if (tm) atomicAdd(&counts[0], tm);
        if (tn) atomicAdd(&counts[1], tn);
        if (tb) atomicAdd(&counts[2], tb);
    }
    __syncthreads();
    for (int o = threadIdx.x; o < kNumOrientations; o += kBlock)
        if (bins[o]) atomicAdd(&obins[o], bins[o]);
}

// The initial state of a directional-solidification domain built on the device
// (TempInit_DirSolidification, SubstrateInit_ConstrainedGrowth, GrainInit and NucleiInit of
// src/CAinitialize.cpp:1025-1055, 1460-1529, 1834-2248): every cell is a wall (the ghost ring and
// the bottom and top planes) or liquid, with its plane's CritTimeStep, LayerID 0 and the Melted
// flag; then the substrate's active cells (GrainIDs 1, 2, ... in list order, cell-centred octahedra
// of half-diagonal 0.01) and the nucleation sites (GrainIDs -1, -2, ... in list order) from the
// host's draws. No cell of such a domain is solid, so GrainInit's last pass (liquid cells without a
// non-solid, non-wall neighbour turn solid) changes nothing when the interior is at least two
// cells wide in x and y.
__global__ __launch_bounds__(kBlock) void k_init_directional(DomainView d, const int32_t *plane_cts, int nx, int ny,
                                                             uint8_t *melted) {
    const Grid gr = grid_of(d);
    for (long long q = static_cast<long long>(blockIdx.x) * kBlock + threadIdx.x; q < d.ncell;
         q += static_cast<long long>(gridDim.x) * kBlock) {
        const Coord c = decode(static_cast<uint32_t>(q), gr);
        const int gx = c.x + d.xoff, gy = c.y + d.yoff;
        const bool wall = gx == -1 || gx == nx || gy == -1 || gy == ny || c.z == 0 || c.z == d.nz - 1;
        const uint8_t ct = wall ? kWall : kLiquid;
        uint4 *r = reinterpret_cast<uint4 *>(d.cells + q);
        r[0] = make_uint4(wall ? kMaskUnknown : 0xFFFFFFFFu, wall ? 0u : kClaimNone, 0u, 0u);
        r[1] = make_uint4(static_cast<uint32_t>(plane_cts[c.z]), 0u, 0u, static_cast<uint32_t>(ct) << 8);
        set_centre(d, q, 0.0, 0.0, 0.0);
        if (melted) melted[q] = wall ? 0 : 1;
    }
}
__global__ __launch_bounds__(kBlock) void k_init_substrate(DomainView d, const uint32_t *cells, uint32_t n) {
    const Grid gr = grid_of(d);
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        const uint32_t q = cells[i];
        const Coord c = decode(q, gr);
        Cell &r = d.cells[q];
        r.lm = kLmUnknown;
        r.dl = 0.01f;
        r.gid = static_cast<int32_t>(i + 1);
        r.ct = kActive | kSeedBit;
        set_centre(d, q, (c.x + d.xoff) + 0.5, (c.y + d.yoff) + 0.5, c.z + 0.5);
        set_alarm(d, 0, q);
    }
}
__global__ __launch_bounds__(kBlock) void k_init_sites(DomainView d, const int32_t *sites, uint32_t n) {
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock)
        d.cells[sites[i]].gid = -static_cast<int32_t>(i + 1);
}

// Initial cell records from the host's compact arrays: no octahedron, no claim, liquid mask not
// yet known; the centres start at zero.
__global__ __launch_bounds__(kBlock) void k_pack(DomainView d, const uint8_t *ct, const int8_t *lid,
                                                 const int32_t *gid, const int32_t *cts) {
    for (long long q = static_cast<long long>(blockIdx.x) * kBlock + threadIdx.x; q < d.ncell;
         q += static_cast<long long>(gridDim.x) * kBlock) {
        uint4 *c = reinterpret_cast<uint4 *>(d.cells + q);
        const bool liquid = (ct[q] & kTypeMask) == kLiquid;
        // a liquid cell: the liquid marker and no claim; any other cell: mask not yet known
        c[0] = make_uint4(liquid ? 0xFFFFFFFFu : kMaskUnknown, liquid ? kClaimNone : 0u, 0u, 0u);
        c[1] = make_uint4(static_cast<uint32_t>(cts[q]), static_cast<uint32_t>(gid[q]), 0u,
                          static_cast<uint32_t>(static_cast<uint8_t>(lid[q])) | (static_cast<uint32_t>(ct[q]) << 8));
        set_centre(d, q, 0.0, 0.0, 0.0);
    }
}

// One per-cell field in the caller's layout (int32 per cell unless noted).
__global__ __launch_bounds__(kBlock) void k_extract(DomainView d, int field, void *out) {
    for (long long q = static_cast<long long>(blockIdx.x) * kBlock + threadIdx.x; q < d.ncell;
         q += static_cast<long long>(gridDim.x) * kBlock) {
        const Cell &c = d.cells[q];
        switch (field) {
        case kFieldCellType: static_cast<int32_t *>(out)[q] = c.ct & kTypeMask; break;
        case kFieldCellTypeRaw: static_cast<uint8_t *>(out)[q] = c.ct; break;  // uint8
        case kFieldGrainId: static_cast<int32_t *>(out)[q] = c.gid; break;
        case kFieldDiagonal: {  // float, with the growth of the steps since the cell was last looked at
            float dl = c.dl;
            if ((c.ct & kTypeMask) == kActive && !(c.lm & kLmUnknown) && !(c.flags & kFresh))
                dl = replay_growth(growth_of(d), dl, static_cast<int>(c.win), growth_index(d, layer_at(d), c.cts, c.lid, static_cast<uint32_t>(q), d.ctl->last_cycle));
            static_cast<float *>(out)[q] = dl;
            break;
        }
        case kFieldCritTimeStep: static_cast<int32_t *>(out)[q] = c.cts; break;
        case kFieldLayerId: static_cast<int32_t *>(out)[q] = c.lid; break;
        case kFieldCentre: {  // float x, y, z
            const Octa &e = d.octa[q];
            float *o = static_cast<float *>(out) + 3 * q;
            o[0] = static_cast<float>(e.x);
            o[1] = static_cast<float>(e.y);
            o[2] = static_cast<float>(e.z);
            break;
        }
        case kFieldCentreF64: {  // double x, y, z, as computed at capture
            const Octa &e = d.octa[q];
            double *o = static_cast<double *>(out) + 3 * q;
            o[0] = e.x;
            o[1] = e.y;
            o[2] = e.z;
            break;
        }
        default: break;
        }
    }
}

// in: n rows of (orientation, cxold, cyold, czold, xp, yp, zp); out: n rows of
// (cx, cy, cz, float(dl), 26 critical lengths recomputed from the new centre).
__global__ __launch_bounds__(kBlock) void k_geometry_probe(const float *guv, const double *in, double *out, int n) {
    const int r = blockIdx.x * kBlock + threadIdx.x;
    if (r >= n) return;
    const double *a = in + 7 * r;
    const float *g = guv + 9 * static_cast<int>(a[0]);
    const Octahedron o = new_octahedron(g, a[1], a[2], a[3], a[4], a[5], a[6]);
    double *b = out + 30 * r;
    b[0] = o.cx;
    b[1] = o.cy;
    b[2] = o.cz;
    b[3] = static_cast<float>(o.dl);
    const Faces f = faces_of(g);
    for (int l = 0; l < 26; l++) b[4 + l] = critical_length(f, a[4], a[5], a[6], o.cx, o.cy, o.cz, nb_dx(l), nb_dy(l), nb_dz(l));
}

// Cells due at the step of that serial, added to *out.
__global__ __launch_bounds__(kBlock) void k_count_due(DomainView d, uint32_t serial, unsigned long long *out) {
    __shared__ unsigned long long sh[kBlock / 64];
    const uint32_t *bits = calendar_slot(d, serial);
    unsigned long long c = 0;
    for (size_t i = static_cast<size_t>(blockIdx.x) * kBlock + threadIdx.x; i < d.nwords;
         i += static_cast<size_t>(gridDim.x) * kBlock)
        c += __builtin_popcount(bits[i]);
    const unsigned long long t = block_sum(c, sh);
    if (threadIdx.x == 0 && t) atomicAdd(out, t);
}

// Unique GrainIDs of a region: the flags k_grain_stats set, counted into *out.
__global__ __launch_bounds__(kBlock) void k_count_flags(const uint32_t *gflag, uint32_t n, unsigned long long *out) {
    __shared__ unsigned long long sh[kBlock / 64];
    unsigned long long c = 0;
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) c += gflag[i] != 0;
    const unsigned long long t = block_sum(c, sh);
    if (threadIdx.x == 0 && t) atomicAdd(out, t);
}

// Fill of n 32-bit words (a kernel rather than a memset node, so that a caller may capture it).
__global__ __launch_bounds__(kBlock) void k_fill(uint32_t *p, size_t n, uint32_t v) {
    for (size_t i = static_cast<size_t>(blockIdx.x) * kBlock + threadIdx.x; i < n;
         i += static_cast<size_t>(gridDim.x) * kBlock)
        p[i] = v;
}

__global__ __launch_bounds__(kBlock) void k_copy(const uint4 *__restrict__ src, uint4 *__restrict__ dst, size_t n) {
    for (size_t i = static_cast<size_t>(blockIdx.x) * kBlock + threadIdx.x; i < n;
         i += static_cast<size_t>(gridDim.x) * kBlock)
        dst[i] = src[i];
}

inline int grid_for(long long n, int cap) {
    long long b = (n + kBlock - 1) / kBlock;
    if (b < 1) b = 1;
    return static_cast<int>(b < cap ? b : cap);
}

}  // namespace

int nucleation_blocks(const DomainView &d) { return grid_for(d.nnuclei, 64); }
int claim_per_cu() {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_claim, kBlock, 0) != hipSuccess) n = 1;
    return n < 1 ? 1 : n;
}
size_t claim_entries(const DomainView &d, uint32_t most_blocks) {
    return static_cast<size_t>(d.units + std::min(d.units, most_blocks)) * kUnitCells;
}
void launch_nucleation(const DomainView &d, const StepAt &at, hipStream_t s) {
    k_nucleate<<<nucleation_blocks(d), kBlock, 0, s>>>(d, at.cycle, at.serial);
}
void launch_capture(const DomainView &d, const StepAt &at, int blocks, hipStream_t s) {
    k_claim<<<blocks, kBlock, 0, s>>>(d, at.cycle, at.serial, at.follows);
    k_apply<<<blocks, kBlock, 0, s>>>(d, at.cycle, at.serial, at.parity);
}
void launch_settle(const DomainView &d, int parity_next, int blocks, hipStream_t s) {
    k_settle<<<blocks, kBlock, 0, s>>>(d, parity_next);
    k_book<<<1, kBlock, 0, s>>>(d, parity_next);
}
void launch_steps(const DomainView &d, int parity, int layer, int steps, bool nucleate, int team, uint64_t launch,
                  hipStream_t s) {
    k_steps<<<team, kTeamBlock, 0, s>>>(d, parity, layer, steps, nucleate ? 1 : 0, launch);
}
void launch_layer_bounds(const DomainView &d, int next_layer, int *out, hipStream_t s) {
    k_layer_bounds<<<grid_for(d.ncell, 4096), kBlock, 0, s>>>(d, next_layer, out);
}
void launch_layer_setup(const DomainView &d, int parity_next, hipStream_t s) {
    const long long n = static_cast<long long>(d.X) * d.Y * (d.nzA - d.zlo);
    k_layer_setup<<<grid_for(n, 4096), kBlock, 0, s>>>(d, parity_next);
}
void launch_rewake(const DomainView &d, int parity_next, int blocks, hipStream_t s) {
    k_rewake<<<blocks, kBlock, 0, s>>>(d, parity_next);
}
void launch_step_timed(const DomainView &d, const StepAt &at, int blocks, hipStream_t s, hipEvent_t *ev) {
    int e = 0;
    auto rec = [&]() { (void)hipEventRecord(ev[e++], s); };
    rec();
    k_nucleate<<<nucleation_blocks(d), kBlock, 0, s>>>(d, at.cycle, at.serial);
    rec();
    rec();
    k_claim<<<blocks, kBlock, 0, s>>>(d, at.cycle, at.serial, at.follows);
    rec();
    rec();
    k_apply<<<blocks, kBlock, 0, s>>>(d, at.cycle, at.serial, at.parity);
    rec();
}
void launch_steps_n(const DomainView *views, const TeamPlace *places, uint32_t workgroups, int steps, int layer,
                    uint64_t launch, hipStream_t s) {
    k_steps_n<<<workgroups, kTeamBlock, 0, s>>>(views, places, layer, steps, launch);
}
void launch_check(const DomainView &d, int cycle, int layer, CheckResult *out, hipStream_t s) {
    k_check<<<grid_for(d.ncell, 4096), kBlock, 0, s>>>(d, cycle, layer, out);
}
void launch_seed_init(const DomainView &d, const uint32_t *cells, uint32_t n, hipStream_t s) {
    k_seed_init<<<grid_for(n, 1024), kBlock, 0, s>>>(d, cells, n);
}
void launch_pack(const DomainView &d, const uint8_t *ct, const int8_t *lid, const int32_t *gid, const int32_t *cts,
                 hipStream_t s) {
    k_pack<<<grid_for(d.ncell, 1 << 16), kBlock, 0, s>>>(d, ct, lid, gid, cts);
}
void launch_grain_stats(const DomainView &d, const uint8_t *melted, const GrainRegion &r, int gmin, uint32_t ngid,
                        uint32_t *gflag, unsigned long long *counts, unsigned int *obins, unsigned int *otop,
                        hipStream_t s) {
    const long long total = static_cast<long long>(r.i1 - r.i0 + 1) * (r.j1 - r.j0 + 1) * (r.k1 - r.k0 + 1);
    k_grain_stats<<<grid_for(total, 2048), kBlock, 0, s>>>(d, melted, r, gmin, ngid, gflag, counts, obins, otop);
}
void launch_init_directional(const DomainView &d, const int32_t *plane_cts, int nx, int ny, uint8_t *melted,
                             const uint32_t *substrate, uint32_t nsub, const int32_t *sites, uint32_t nsites,
                             hipStream_t s) {
    k_init_directional<<<grid_for(d.ncell, 1 << 16), kBlock, 0, s>>>(d, plane_cts, nx, ny, melted);
    if (nsub) k_init_substrate<<<grid_for(nsub, 4096), kBlock, 0, s>>>(d, substrate, nsub);
    if (nsites) k_init_sites<<<grid_for(nsites, 4096), kBlock, 0, s>>>(d, sites, nsites);
}
void launch_extract(const DomainView &d, int field, void *out, hipStream_t s) {
    k_extract<<<grid_for(d.ncell, 1 << 16), kBlock, 0, s>>>(d, field, out);
}
void launch_count_flags(const uint32_t *gflag, uint32_t n, unsigned long long *out, hipStream_t s) {
    k_count_flags<<<grid_for(n, 1024), kBlock, 0, s>>>(gflag, n, out);
}
void launch_count_due(const DomainView &d, uint32_t serial, unsigned long long *out, hipStream_t s) {
    k_count_due<<<grid_for((d.ncell + 31) / 32, 1024), kBlock, 0, s>>>(d, serial, out);
}
void launch_fill(uint32_t *p, size_t n, uint32_t v, hipStream_t s) {
    k_fill<<<grid_for(static_cast<long long>(n), 4096), kBlock, 0, s>>>(p, n, v);
}
void launch_copy(const uint4 *src, uint4 *dst, size_t n, hipStream_t s) {
    k_copy<<<grid_for(static_cast<long long>(n), 1 << 16), kBlock, 0, s>>>(src, dst, n);
}
void launch_geometry_probe(const float *guv, const double *in, double *out, int n, hipStream_t s) {
    k_geometry_probe<<<grid_for(n, 1 << 20), kBlock, 0, s>>>(guv, in, out, n);
}

}  // namespace exaca
