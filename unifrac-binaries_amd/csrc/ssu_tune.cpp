#include "ssu_tune.hpp"

#include <algorithm>
#include <cmath>

namespace ssu {

namespace {

// Marginal seconds per unit on one MI355X, fitted to whole-plan timings at
// three thresholds each on the 16,384-sample (100k tips) and 8,192-sample
// (50k tips) workloads (total = fixed + terms * term + postings * posting); the
// modelled optimum lands within the measured one for every kind (weighted
// 0.193 vs 0.2, FP64 weighted 0.24 vs 0.23 - 0.3, generalized 0.38 vs 0.4,
// Gram 0.07 vs 0.06 - 0.1).  The per-term cost includes the list building
// and row lists, whose work follows the postings.
struct Rates {
    double term;      // one (pair, node) term of the tiled kernel; Gram: one (pair, column) unit
    double posting;   // one posting visited by the row walk
    double onesided = 0.0;   // VAW: one (posting slot, total) one-sided term
};

Rates rates_of(SplitKind k, double alpha) {
    switch (k) {
    // 16,384 samples, theta 0.14 .. 0.26: tiles 70.1 .. 42.6 ms, posting phase 29.1 .. 56.5 ms,
    // device total 115.1, 111.6 (0.17), 111.2 (0.2), 112.5 (0.23), 115.0 ms
    case SplitKind::weighted32: return {3.3e-14, 8.9e-13};
    // 3,001 samples (20k tips), theta 0.1 / 0.23 / 0.4: tiles 2.91 / 1.62 / 1.01 ms, posting
    // phase 0.54 / 1.09 / 1.96 ms, device total 4.20 / 3.46 / 3.73 ms (0.3: 3.50)
    case SplitKind::weighted64: return {8.2e-14, 1.42e-12};
    // 4,000 samples (20k tips), theta 0.2 .. 0.6: tiles 8.29 .. 3.03 ms (alpha 1/2: reciprocal
    // square roots), 9.94 .. 3.74 (0.3: log2 and exp2), 3.14 .. 1.14 (1: no power), posting
    // phase 1.73 .. 6.20 ms; best totals at 0.4 (9.39 ms), 0.5 (10.5) and 0.2 - 0.3 (5.9)
    case SplitKind::generalized32: return {alpha == 1.0 ? 8.5e-14 : alpha == 0.5 ? 2.25e-13 : 2.65e-13, 1.57e-12};
    // Gram: 0.82 ms for the 2.96e11 units of 8,000 samples, 3.73 for the 1.21e12 of 16,384
    case SplitKind::gram: return {2.9e-15, 6.1e-13};
    // FP64 generalized, 1,200 samples, theta 0.2 .. 0.6: alpha 1/2 tiles 2.54 .. 0.90 ms, posting
    // phase 0.58 .. 1.55 (totals 3.51, 2.83 at 0.4 - 0.6); other alpha (an FP64 power per tile
    // term, two per posting) 8.07 .. 2.84 and 1.01 .. 3.28 (totals 9.47, 6.5 at 0.6); alpha 1
    // takes no power on the tiles
    case SplitKind::generalized64:
        if (alpha == 0.5) return {6.7e-13, 3.8e-12};
        return {alpha == 1.0 ? 2.0e-13 : 2.15e-12, 8.8e-12};
    // VAW: the tiles' term; a posting (three FP64 reciprocal square roots); a one-sided term at
    // one total (or point).  4,000 samples, theta 0.2 .. 0.8: tiles 9.37 .. 2.09 ms, posting phase
    // 2.78 .. 14.3 (totals 14.3, 13.2 at 0.3, 13.5 at 0.4, 18.5); FP64, 2,000 samples: 6.42 .. 1.67
    // and 1.28 .. 5.90 (sums at few points: 8.63, 7.48 at 0.4, 8.49; 1,500 samples at every total:
    // 5.42 at 0.2, 5.19 at the model's 0.29, 5.43 at 0.42); the one-sided rate from the sums at every total
    // of the 8,192-sample workload.  Weighted and presence terms are within 15% of each other; the
    // weighted rates are used for both
    case SplitKind::vaw32: return {2.65e-13, 2.37e-12, 4.13e-13};
    case SplitKind::vaw64: return {6.7e-13, 3.8e-12, 6.2e-13};
    }
    return {1.0, 1.0};
}

}  // namespace

SplitChoice choose_split(SplitKind kind, uint32_t n, const std::vector<uint32_t>& occupancy, uint64_t max_slots,
                         uint32_t cols, double alpha) {
    SplitChoice best;
    if (n < 2 || occupancy.empty()) return best;
    const Rates r = rates_of(kind, alpha);
    // nodes by occupancy (0: held by no sample, no cost either way); an
    // occupancy above n (never, for counts of n samples) counts as n
    std::vector<uint64_t> hist((size_t)n + 1, 0);
    for (uint32_t x : occupancy) ++hist[std::min(x, n)];
    // cost with every node on the tiles; then move nodes to the posting lists in
    // increasing occupancy (thr = c + 1 moves every node held by at most c samples)
    const double pairs = 0.5 * (double)n * n;   // a node on the tiles costs every pair
    double tiles = 0.0;
    for (uint32_t c = 1; c <= n; ++c) tiles += (double)hist[c] * pairs * r.term;
    best.model_ms_none = best.model_ms = tiles * 1e3;
    double cost = tiles, posts = 0.0;
    uint64_t slots = 0;
    for (uint32_t c = 0; c <= n; ++c) {
        if (!hist[c]) continue;
        if (c > 0) {
            const double m = (double)hist[c], x = c;
            cost -= m * pairs * r.term;
            posts += m * (0.5 * x * (x - 1.0) * r.posting + x * (double)cols * r.onesided);
            slots += hist[c] * c;
        }
        if (slots >= max_slots) break;
        if (cost + posts < best.model_ms * 1e-3) {
            best.model_ms = (cost + posts) * 1e3;
            best.thr = c + 1;
        }
    }
    return best;
}

}  // namespace ssu
