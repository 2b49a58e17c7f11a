// growth.hpp -- the half-diagonal growth recurrence of a CA cell, advanced many steps at once.
//
// Each executed step past a cell's liquidus time stores dl = float(double(dl) + g_k)
// (src/CAupdate.cpp:257-261). On the table's plateau (the 0.045 cap) g is a constant c. For dl a
// positive normal float in the binade [2^(e-1), 2^e), dl is a multiple of u = 2^(e-24), and the
// double sum dl + c rounds to float the same way for every such dl: the sum's bits below u come
// from c alone, at the same double precision across the binade. Unless that rounding is a tie,
// every step inside the binade therefore adds the same delta, and the interior of a binade is
// crossed in one jump. Steps next to a binade boundary, ties and non-normal values are taken one at
// a time. Host and device share these functions; the host copy is what the tests check against
// the step-by-step recurrence.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <vector>

namespace exaca {

__host__ __device__ inline float grow_step(float x, double g) {
    return static_cast<float>(static_cast<double>(x) + g);
}

__host__ __device__ inline uint32_t float_bits(float x) { return __builtin_bit_cast(uint32_t, x); }

// e with 2^(e-1) <= x < 2^e for a positive normal float.
__host__ __device__ inline int binade_of(float x) { return static_cast<int>((float_bits(x) >> 23) & 0xFFu) - 126; }

// Whether the step x -> y = grow_step(x, c) gives the constant delta of x's binade; if so, delta
// and the number of further steps from y whose results stay two steps clear of the binade's top.
__host__ __device__ inline bool binade_run(float x, float y, double c, double &delta, int &room) {
    const uint32_t be = (float_bits(x) >> 23) & 0xFFu;
    if ((float_bits(x) >> 31) || be == 0 || be == 0xFFu) return false;
    const int e = binade_of(x);
    if (binade_of(y) != e) return false;
    const double u = std::ldexp(1.0, e - 24);
    if (std::fabs((static_cast<double>(x) + c) - static_cast<double>(y)) == 0.5 * u) return false;  // tie
    delta = static_cast<double>(y) - static_cast<double>(x);
    if (!(delta > 0)) return false;
    const double r = std::floor((std::ldexp(1.0, e) - 2.0 * delta - static_cast<double>(y)) / delta) - 1.0;
    room = r > 0 ? (r < 1.0e9 ? static_cast<int>(r) : 1000000000) : 0;
    return true;
}

// x after n steps of the constant increment c.
__host__ __device__ inline float advance_const(float x, int n, double c) {
    while (n > 0) {
        const float y = grow_step(x, c);
        n--;
        double delta = 0;
        int room = 0;
        if (n == 0 || !binade_run(x, y, c, delta, room)) {
            x = y;
            continue;
        }
        const int m = room < n ? room : n;
        x = static_cast<float>(static_cast<double>(y) + m * delta);
        n -= m;
    }
    return x;
}

// First n in 1 .. horizon at which x after n steps of the constant increment c reaches thr;
// horizon when it does not.
__host__ __device__ inline int reach_const(float x, double c, float thr, int horizon) {
    int n = 0;
    while (n < horizon) {
        const float y = grow_step(x, c);
        n++;
        if (y >= thr) return n;
        double delta = 0;
        int room = 0;
        if (n == horizon || !binade_run(x, y, c, delta, room)) {
            x = y;
            continue;
        }
        const int m = room < horizon - n ? room : horizon - n;
        // the values after further steps are y + i delta (i = 1 .. m), all exact in double
        const double yd = static_cast<double>(y), t = static_cast<double>(thr);
        double need = std::ceil((t - yd) / delta);
        if (need < 1) need = 1;
        if (need <= m) {
            int i = static_cast<int>(need);
            while (i > 1 && yd + (i - 1) * delta >= t) i--;
            while (yd + i * delta < t) i++;
            return n + i;
        }
        x = static_cast<float>(yd + m * delta);
        n += m;
    }
    return horizon;
}

// ---- Any run of table entries at once. Inside a binade the delta of the entry g_k is the same for
// every dl there (ties apart), so in units u of the binade the half-diagonal is an integer that
// grows by whole numbers D_k, and their prefix sums give it after any number of steps: two reads
// instead of one rounding after another (63 steps of them took a cell's lane 10 us). A row holds
// one binade's sums of D_1 .. D_k for k = 0 .. ksat and, last, the plateau's delta: the increment of
// every k >= ksat. Rows of binades where an entry ties are marked unusable. ----
constexpr int kSumLo = -6, kSumHi = 3;  // binades [2^(e-1), 2^e) with rows: half-diagonals 2^-7 .. 8
constexpr int kSumRows = kSumHi - kSumLo + 1;
constexpr uint32_t kMantissaEnd = 1u << 24;  // mantissas, in units of the binade, lie below this
constexpr int kSumSpan = 128;                // most steps taken at once: the sums are modulo 2^32
constexpr int kSumMost = 1 << 18;            // longest table with rows
// The row of binade e: most half-diagonals that still grow lie in [1, 2), [2, 4) and [1/2, 1), whose rows
// come first (a kernel stages the first few in LDS).
__host__ __device__ inline int sum_row(int e) {
    return static_cast<int>((0x3102456789ull >> (4 * (e - kSumLo))) & 15u);
}

struct GrowthSums {
    std::vector<uint32_t> sums;  // kSumRows rows of ksat + 2
    uint32_t usable = 0;         // bit r: row r holds for every dl of its binade
};
inline GrowthSums growth_sums(const std::vector<double> &grow, int ksat) {
    GrowthSums s;
    const size_t len = static_cast<size_t>(ksat) + 2;
    s.sums.assign(kSumRows * len, 0u);
    if (ksat > kSumMost) {
        s.sums.assign(1, 0u);
        return s;
    }
    for (int e = kSumLo; e <= kSumHi; e++) {
        const int r = sum_row(e);
        uint32_t *row = &s.sums[r * len], sum = 0;
        bool tie = false;
        for (int k = 1; k <= ksat + 1; k++) {
            const double g = k < ksat ? grow[k] : grow.back();
            // dl + g is rounded to a multiple of 2^(e-53), then to one of u = 2^(e-24)
            const double q = std::ldexp(std::rint(std::ldexp(g, 53 - e)), -29);
            tie |= q - std::floor(q) == 0.5;
            const uint32_t delta = static_cast<uint32_t>(std::min(std::rint(q), static_cast<double>(kMantissaEnd)));
            if (k <= ksat) row[k] = (sum += delta);
            else row[ksat + 1] = delta;
        }
        if (!tie) s.usable |= 1u << r;
    }
    return s;
}

// A row's sums: p[k] up to the plateau, from there on the plateau's delta each step. P: a pointer to the
// row, in whatever memory it lies.
template <typename P>
struct SumRow {
    P p;
    int ksat;
    uint32_t plateau;
    __host__ __device__ uint32_t at(int k) const {
        const int i = k < ksat ? k : ksat;
        return p[i] + static_cast<uint32_t>(k - i) * plateau;
    }
};
template <typename P>
__host__ __device__ inline SumRow<P> sum_row_at(P row, int ksat) {
    return SumRow<P>{row, ksat, row[ksat + 1]};
}

// t: the table. ksat, gsat; inc(k): the increment of step k; usable; with_row(r, f): calls f with the
// SumRow of row r.
template <typename T>
__host__ __device__ inline int usable_row(const T &t, float x) {
    const int e = binade_of(x);  // a sign bit falls out of it, so it is tested
    if (!(x > 0) || e < kSumLo || e > kSumHi) return -1;
    const int r = sum_row(e);
    return (t.usable >> r) & 1u ? r : -1;
}
__host__ __device__ inline uint32_t mantissa_of(float x) { return (float_bits(x) & 0x7FFFFFu) | 0x800000u; }
__host__ __device__ inline float with_mantissa(float x, uint32_t m) {
    return __builtin_bit_cast(float, (float_bits(x) & 0x7F800000u) | (m & 0x7FFFFFu));
}
// Where a search between lo and hi looks for the place of lim next: where a straight line from vlo to
// vhi reaches it, strictly between them. Any answer is right; a close one ends the search soon (the
// increments change little over a run, and not at all on the plateau).
__host__ __device__ inline int probe(int lo, int hi, uint32_t vlo, uint32_t vhi, uint32_t lim) {
    const float num = static_cast<float>(lim - vlo) * static_cast<float>(hi - lo);
#ifdef __HIP_DEVICE_COMPILE__
    const float q = num * __builtin_amdgcn_rcpf(static_cast<float>(vhi - vlo));
#else
    const float q = num / static_cast<float>(vhi - vlo);
#endif
    const int mid = lo + static_cast<int>(q < 1024.0f ? q : 1024.0f);
    return mid <= lo ? lo + 1 : (mid >= hi ? hi - 1 : mid);
}
// The last of 0 .. hi after which the sum is below lim: m + row(k + i) - row(k) is below lim at 0 and
// not at hi. at: the sum there.
template <typename R>
__host__ __device__ inline int last_below(const R &row, int k, uint32_t base, uint32_t m, int hi, uint32_t vhi,
                                          uint32_t lim, uint32_t &at) {
    int lo = 0;
    at = m;
    for (int turn = 0; hi - lo > 1; turn++) {
        // along the line, next to the bracket's nearer end, along the line again, then halves
        const int mid = turn > 2 ? (lo + hi) >> 1 : (turn == 1 ? (lo > 0 ? lo + 1 : hi - 1) : probe(lo, hi, at, vhi, lim));
        const uint32_t v = m + (row.at(k + mid) - base);
        if (v < lim) {
            lo = mid;
            at = v;
        }
        else {
            hi = mid;
            vhi = v;
        }
    }
    return lo;
}

// x after the growth of the steps k0 + 1 .. k1.
template <typename T>
__host__ __device__ inline float advance_steps(const T &t, float x, int k0, int k1) {
    while (k0 < k1) {
        const int r = usable_row(t, x);
        if (r >= 0 && k1 - k0 <= kSumSpan) {
            t.with_row(r, [&](const auto &row) {
                const uint32_t m = mantissa_of(x), base = row.at(k0);
                const uint32_t all = m + (row.at(k1) - base);
                if (all < kMantissaEnd) {
                    x = with_mantissa(x, all);
                    k0 = k1;
                }
                else {  // to the last step that stays in the binade; the one after it is taken by itself
                    uint32_t at;
                    k0 += last_below(row, k0, base, m, k1 - k0, all, kMantissaEnd, at);
                    x = with_mantissa(x, at);
                }
            });
            if (k0 == k1) return x;
        }
        else if (k0 + 1 >= t.ksat)
            return advance_const(x, k1 - k0, t.gsat);
        x = grow_step(x, t.inc(++k0));
    }
    return x;
}

// First n in 1 .. horizon at which x, now at step k, reaches thr after n more steps; horizon when it
// does not.
template <typename T>
__host__ __device__ inline int reach_steps(const T &t, float x, int k, float thr, int horizon) {
    int n = 0;
    while (n < horizon) {
        const int r = usable_row(t, x);
        if (r >= 0 && horizon - n <= kSumSpan) {
            int found = 0;
            t.with_row(r, [&](const auto &row) {
                const uint32_t m = mantissa_of(x), base = row.at(k + n);
                const int et = binade_of(thr), ex = binade_of(x);
                // thr in the binade's units, or the binade's end when it lies beyond
                const uint32_t lim = !(thr > 0) || et < ex ? 0u : (et > ex ? kMantissaEnd : mantissa_of(thr));
                const uint32_t all = m + (row.at(k + horizon) - base);
                if (all < lim)
                    found = horizon;
                else if (m >= lim)
                    found = n + 1;
                else {
                    uint32_t at;
                    const int lo = last_below(row, k + n, base, m, horizon - n, all, lim, at);
                    if (lim < kMantissaEnd)
                        found = n + lo + 1;
                    else {
                        x = with_mantissa(x, at);
                        n += lo;
                    }
                }
            });
            if (found) return found;
        }
        else if (k + n + 1 >= t.ksat)
            return n + reach_const(x, t.gsat, thr, horizon - n);
        n++;
        x = grow_step(x, t.inc(k + n));
        if (x >= thr) return n;
    }
    return horizon;
}

}  // namespace exaca
