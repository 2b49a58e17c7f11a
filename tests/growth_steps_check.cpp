// Checks the growth over any run of table entries (advance_steps and reach_steps of
// exaca_amd/csrc/growth.hpp, prefix sums per binade) against one float rounding per step: growth
// tables of the shape the solver builds (a rising polynomial of a float-accumulated undercooling with
// zeros below and the 0.045 cap above), of equal entries, of one entry, and with entries that tie in
// some binades; half-diagonals at random, next to powers of two, subnormal and outside the
// rows' range; runs across the plateau's start and longer than a row may take at once. Prints the
// number of mismatches and exits nonzero on any.
#include <cstdio>
#include <random>

#include "growth.hpp"

using namespace exaca;

struct Table {
    std::vector<double> grow;
    int ksat = 0;
    double gsat = 0;
    GrowthSums s;
    uint32_t usable = 0;
    explicit Table(std::vector<double> g) : grow(std::move(g)) {
        ksat = static_cast<int>(grow.size()) - 1;
        while (ksat > 0 && grow[ksat - 1] == grow.back()) ksat--;
        gsat = grow.back();
        s = growth_sums(grow, ksat);
        usable = s.usable;
    }
    double inc(int k) const { return k < ksat ? grow[k] : gsat; }
    template <typename F>
    void with_row(int r, F &&f) const {
        f(sum_row_at(&s.sums[static_cast<size_t>(r) * (ksat + 2)], ksat));
    }
};

int main() {
    std::mt19937_64 gen(2024);
    std::uniform_real_distribution<double> u01(0.0, 1.0);
    std::vector<Table> tables;
    for (double dU : {0.02, 0.1, 0.7, 5.0}) {
        std::vector<double> g;
        float u = 0;
        while (u < 210.0f) {
            const double lu = u;
            double v = -7.5e-8 * lu * lu * lu + 2.4e-5 * lu * lu - 2.0e-4 * lu;
            v = v < 0 ? 0 : v;
            g.push_back(v < 0.045 ? v : 0.045);
            u += static_cast<float>(dU);
        }
        tables.emplace_back(g);
    }
    tables.emplace_back(std::vector<double>(40, 0.045));
    tables.emplace_back(std::vector<double>(1, 0.0));
    std::vector<double> ties;
    for (int k = 0; k < 300; k++) ties.push_back((k % 37 + 0.5) * std::ldexp(1.0, -23 + k % 3));
    tables.emplace_back(ties);
    std::vector<double> big;
    for (int k = 0; k < 200; k++) big.push_back(0.0449 * u01(gen));
    tables.emplace_back(big);
    long long cases = 0, bad = 0, rows = 0;
    for (const Table &t : tables) rows += __builtin_popcount(t.usable);
    for (int i = 0; i < 600000; i++) {
        const Table &t = tables[i % tables.size()];
        float x;
        if (i % 5 == 0) {
            x = std::nextafter(static_cast<float>(std::ldexp(1.0, static_cast<int>(u01(gen) * 14) - 9)), 0.0f);
            for (int k = static_cast<int>(u01(gen) * 40); k > 0; k--) x = std::nextafter(x, 0.0f);
        }
        else if (i % 97 == 1)
            x = i % 2 ? 1e-39f : 0.0f;
        else
            x = static_cast<float>(std::exp(std::log(1e-3) + u01(gen) * (std::log(20.0) - std::log(1e-3))));
        const int k0 = static_cast<int>(u01(gen) * (t.ksat + 80));
        const int n = i % 50 == 7 ? static_cast<int>(u01(gen) * 400) : static_cast<int>(u01(gen) * 66);
        float ref = x;
        for (int k = 1; k <= n; k++) ref = grow_step(ref, t.inc(k0 + k));
        const float got = advance_steps(t, x, k0, k0 + n);
        cases++;
        if (float_bits(ref) != float_bits(got)) {
            if (bad++ < 5) printf("advance x=%.9g k0=%d n=%d: %.9g, stepwise %.9g\n", x, k0, n, got, ref);
        }
        const float thr = i % 31 == 5 ? __builtin_inff()
                          : i % 3     ? static_cast<float>(x + u01(gen) * 0.06 * 63)
                                      : static_cast<float>(ref + (u01(gen) - 0.5) * 1e-6);
        const int horizon = i % 19 == 2 ? 1 + static_cast<int>(u01(gen) * 200) : 63;
        int want = horizon;
        float y = x;
        for (int m = 1; m <= horizon; m++) {
            y = grow_step(y, t.inc(k0 + m));
            if (y >= thr) {
                want = m;
                break;
            }
        }
        const int have = reach_steps(t, x, k0, thr, horizon);
        cases++;
        if (want != have) {
            if (bad++ < 5) printf("reach x=%.9g k0=%d thr=%.9g horizon=%d: %d, stepwise %d\n", x, k0, thr, horizon, have, want);
        }
    }
    printf("cases %lld usable rows %lld mismatches %lld\n", cases, rows, bad);
    return bad || rows < 50 ? 1 : 0;
}
