// Which tiles a grouped product of an expert layer runs on (host code, no HIP).
#pragma once

#include <cmath>

namespace paras {

constexpr int kFormStep = 64;                           // contraction steps of a turn
constexpr int kSuperM = 8, kSuperN = 4;             // row tiles and column units of a super-tile (grouped_gemm_direct_kernel)

// The tiles of a grouped product: rows, weight rows, stages, workgroups a CU holds, and for the gate-up product and the plain one the time
// in us of 64 contraction steps on a CU that is full (`step`) and at least (`lat`).  The last two are grouped_gemm_direct_kernel, its tiles dealt in
// super-tiles or one by one.
struct GroupedForm { int m, n, stages, per_cu; double step[2], lat[2]; };
inline constexpr GroupedForm kForms[] = {{128, 128, 2, 2, {0.91, 0.78}, {0.66, 0.47}}, {128, 128, 3, 1, {0.54, 0.36}, {0.13, 0.02}}, {64, 128, 2, 3, {0.74, 0.33}, {0.51, 0.42}},
                                         {64, 128, 4, 1, {0.19, 0.24}, {0.35, 0.23}}, {32, 128, 4, 2, {0.30, 0.07}, {0.15, 0.16}}, {256, 256, 2, 1, {1.13, 0.97}, {0.32, 0.30}},
                                         {256, 256, 2, 1, {1.13, 0.97}, {0.32, 0.30}}};
constexpr int kFormCount = sizeof(kForms) / sizeof(kForms[0]), kDirectForm = kFormCount - 2, kOneByOne = kFormCount - 1;

// Tiles of 256 rows where each of E experts has R / E rows on average and each row is sent on its own (a normal distribution).
inline double tiles_256(long E, long R) {
    const double rows = static_cast<double>(R) / E, spread = std::sqrt(2.0 * rows);
    double n = 1.0 - std::exp(-rows);
    for (double j = 256; j < rows + 3 * spread; j += 256) n += 0.5 * std::erfc((j + 0.5 - rows) / spread);
    return E * n;
}

// The least estimated time, from three that overlap for the most part (the fourth root of the sum of their fourth powers): rounds of
// workgroups times their contraction and stores, the way of the weights from memory, and that of all tiles' operands from the caches.  (How
// the rows are spread over the experts is known on the device only: half an empty tile per expert, one tile where an expert has less than two
// thirds of one.)  Fitted to 1800 timings of 150 layers (8 to 8192 tokens, 4 to 64 experts, H 512 to 4096, I 512 to 14336), over which the
// choice is 2 % (gate-up) and 5 % (down) slower than the best form in the mean; always the same form is 15 % and 22 % at the least.
//   256 x 256 tiles one by one are looked at for up to three rounds: of more the last is a small part.  One tile too many is a round, so their number is estimated by
// the spread of the rows (a last round of 2 % is most often none), and a round is taken 5 % and 6 us longer than the contraction and stores.  Against super-tiles, which the line above gives half a
// tile per expert too many, the same number counts, less 0.7 (the last tile an expert sends may be short): 5916 tokens, top-2, 8 experts, H 3264, I 12736, down, three rounds
// either way, one by one 61 us more.  Against smaller tiles, of which a CU holds two or three that hide each other's starts and ends, two and three rounds have to be a
// sixth ahead: gate-up of 5171 tokens, top-2, 8 experts, 1408 x 1152 14 us more, down of 1657 tokens, top-4, 32 experts, 2112 x 2688 (1.1 rounds) 22.  Over 450 products of
// 130 layers, each both ways, it is chosen for 32: none over 0.6 % of its layer slower than without this form, the mean
// 8.5 % faster.
inline int grouped_form(bool swiglu, long E, long R, long N, long K) {
    const int w = swiglu ? 0 : 1;
    const double start = swiglu ? 3.9 : 1.3, store = swiglu ? 15.4 : 9.4, rows = static_cast<double>(R) / E, used = R < E ? R : E;
    const double memory = used * N * K * (swiglu ? 4.0 / 5.34e6 : 2.0 / 5.37e6), cached = swiglu ? 16.4e6 : 14.1e6;
    auto fourth = [](double v) { return v * v * v * v; };
    int best = 0;
    double best_cost = 1e300, direct_rest = 0.0;
    for (int f = 0; f < kFormCount; ++f) {
        const GroupedForm& t = kForms[f];
        const long cols = swiglu ? t.n / 2 : t.n, units = (N + cols - 1) / cols, k_tiles = K / kFormStep, turns = (k_tiles + t.stages - 1) / t.stages * t.stages;
        if (f == kOneByOne && static_cast<double>(R) / 256 * units > 3 * 256) continue;
        const double m_tiles = f == kOneByOne ? tiles_256(E, R) : rows < 0.7 * t.m ? used : E * (rows / t.m + 0.5), tiles = m_tiles * units;
        auto round = [&](double n) {
            const double c = t.step[w] * n / t.per_cu;
            return turns * (c > t.lat[w] ? c : t.lat[w]) + start + store * t.m * cols / 65536.0 * n;
        };
        auto supers = [&](double m) {    // super-tiles of 32 workgroups, dealt to the 8 XCDs
            return std::ceil(std::ceil(m / kSuperM) * std::ceil(static_cast<double>(units) / kSuperN) / 8) * round(1.0);
        };
        const double traffic = tiles * (t.m + t.n) * K * 2.0 / cached;
        double us, ahead = 1.0;
        if (f == kDirectForm) {
            us = supers(m_tiles);
            direct_rest = fourth(memory) + fourth(traffic);
        } else if (f == kOneByOne) {
            const double rounds = std::fmax(std::ceil(tiles / 256 - 0.02), 1.0);
            us = 1.05 * rounds * (round(1.0) + 6.0);
            if (best == kDirectForm) best_cost = std::fmin(best_cost, fourth(supers(std::fmax(m_tiles - 0.7, 1.0))) + direct_rest);
            else if (rounds > 1)     ahead = 7.0 / 6;
        } else {
            const double slots = 256.0 * t.per_cu, full = std::floor(tiles / slots), rest = std::ceil((tiles - full * slots) / 256.0);
            us = full * round(t.per_cu) + (rest > 0 ? round(rest) : 0.0);
        }
        const double cost = (fourth(us) + fourth(memory) + fourth(traffic)) * fourth(ahead);
        if (cost < best_cost) {
            best_cost = cost;
            best = f;
        }
    }
    return best;
}

}  // namespace paras
