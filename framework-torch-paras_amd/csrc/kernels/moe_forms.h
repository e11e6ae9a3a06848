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

// All tiles of the grouped products: those above in their order, then what grouped_tile_kernel has besides.  (A time of zero: not for that product.)
inline constexpr GroupedForm kAllForms[] = {{128, 128, 2, 2, {0.519, 0.476}, {0.607, 0.611}}, {128, 128, 3, 1, {0.312, 0.306}, {0.164, 0.131}},
                                             {64, 128, 2, 3, {0.594, 0.789}, {0.472, 0.526}}, {64, 128, 4, 1, {0.183, 0.227}, {0.215, 0.251}},
                                             {32, 128, 4, 2, {0.372, 0.042}, {0.218, 0.461}}, {256, 256, 2, 1, {0.614, 0.812}, {0.539, 0.137}},
                                             {256, 256, 2, 1, {0.767, 0.288}, {0.403, 0.706}}, {32, 64, 4, 3, {0.256, 0.409}, {0.211, 0.204}},
                                             {64, 64, 4, 2, {0.229, 0.318}, {0.211, 0.224}}, {96, 64, 4, 2, {0.201, 0.181}, {0.286, 0.377}},
                                             {96, 128, 2, 2, {0.478, 0.601}, {0.545, 0.547}}, {192, 128, 2, 2, {0.453, 0.788}, {0.737, 0.663}},
                                             {160, 128, 2, 2, {0.696, 0.0}, {0.575, 0.0}}, {192, 256, 2, 1, {0.0, 0.636}, {0.0, 0.574}},
                                             {128, 256, 3, 1, {0.0, 0.533}, {0.0, 0.223}}};
constexpr int kAllFormCount = sizeof(kAllForms) / sizeof(kAllForms[0]);

// Tiles of m rows, as tiles_256; where an expert fills more than six, half a tile each is what is lost.
inline double tiles_of_rows(long E, long R, int m) {
    const double rows = static_cast<double>(R) / E;
    if (rows > 6.0 * m) return E * (rows / m + 0.5);
    const double spread = std::sqrt(2.0 * rows);
    double n = 1.0 - std::exp(-rows);
    for (double j = m; j < rows + 3 * spread; j += m) n += 0.5 * std::erfc((j + 0.5 - rows) / spread);
    return E * n;
}

// The tiles that a product runs on: the least estimated time, as above, of all forms, of grouped_gemm_direct_kernel's two dealings the one that grouped_form
// takes, and none where it takes neither.  The number of an expert's tiles is a matter of chance, and one tile more can be a round more: the time is a mean over the
// expected number and half a tile per square root of an expert less and more.  grouped_form's own choice stays unless another one is estimated to be a tenth (gate-up) or a
// sixteenth (down) faster.  Fitted to 50000 timings of 1806 layers (4 to 64 experts, 8 to 16384 routed rows, H 512 to 4096, I 512 to
// 14336, weights from HBM): 2.0 % (gate-up) and 2.3 % (down) of a layer's time faster in the mean than grouped_form alone, 7.5 % and 4.2 % where the choice is another one; 7
// and 8 layers are more than 4 % slower, of what was measured another 1.9 % and 0.9 % could be had.  What the further forms bring.  32 x 64 with four stages, three to a CU, is for
// products whose tiles are too few for 256 CUs: down of 230 tokens, top-2, 8 experts, 640 x 4096, 26.8 us on 32 x 128, 19.5.  192 x 128 and 160 x 128 with two stages,
// two to a CU, hide each other's SwiGLU and stores, which 256 x 256 tiles do one CU at a time, and waste less of an expert's last tile: gate-up of 2167 tokens,
// top-4, 32 experts, 1856 x 1280, 181 us on 256 x 256, 166.  192 x 256 and 128 x 256: down of 1156 tokens, top-2, 8 experts, 3520 x 14272, and of 910,
// 3008 x 10496 (with the gate-up product's change layers 1201 -> 860 and 596 -> 467).  Where the tiles are about as many as the CUs hold, chance decides: gate-up of 3221 tokens, top-2, 8
// experts, 1088 x 832 came to 520 tiles of 192 x 128 for 512 places, layer 75 -> 93.
inline int grouped_tiles(bool swiglu, long E, long R, long N, long K) {
    const int w = swiglu ? 0 : 1, base = grouped_form(swiglu, E, R, N, K);
    const double start = swiglu ? 1.460 : 0.634, store = swiglu ? 30.08 : 7.54, beside = swiglu ? 0.586 : 0.601;          // us; `beside`: with other workgroups on the CU
    const double from_memory = swiglu ? 20.11e6 : 22595.85e6, from_caches = swiglu ? 30.70e6 : 458704.40e6;                 // bytes per us
    const double supers = swiglu ? 0.995 : 0.838, one_by_one = swiglu ? 1.010 : 0.666, ahead = swiglu ? 0.90 : 0.94;
    const double memory = static_cast<double>(R < E ? R : E) * N * K * (swiglu ? 4.0 : 2.0) / from_memory, chance = 0.5 * std::sqrt(static_cast<double>(E));
    auto fourth = [](double v) { return v * v * v * v; };
    double by_rows[9] = {};           // row tiles of 32, 64 ... 256
    int best = 0;
    double best_cost = 1e300;
    for (int f = 0; f < kAllFormCount; ++f) {
        const GroupedForm& t = kAllForms[f];
        const bool direct = f == kDirectForm || f == kOneByOne;
        if (t.step[w] == 0.0 || (direct && f != base)) continue;
        const long cols = swiglu ? t.n / 2 : t.n, units = (N + cols - 1) / cols, k_tiles = K / kFormStep, turns = (k_tiles + t.stages - 1) / t.stages * t.stages;
        double& m_tiles = by_rows[t.m / 32];
        if (m_tiles == 0.0) m_tiles = tiles_of_rows(E, R, t.m);
        const double stores = store * t.m * cols / 65536.0 * (t.per_cu > 1 ? beside : 1.0), slots = 256.0 * t.per_cu;
        auto round = [&](double n) {
            const double c = t.step[w] * n / t.per_cu;
            return turns * (c > t.lat[w] ? c : t.lat[w]) + start + stores * n;
        };
        const double one_round = round(t.per_cu);
        auto rounds = [&](double m) {
            if (f == kDirectForm) return supers * std::ceil(std::ceil(m / kSuperM) * std::ceil(static_cast<double>(units) / kSuperN) / 8) * one_round;
            if (f == kOneByOne) return one_by_one * std::ceil(m * units / 256) * one_round;
            const double full = std::floor(m * units / slots), rest = std::ceil((m * units - full * slots) / 256.0);
            return full * one_round + (rest > 0 ? round(rest) : 0.0);
        };
        const double us = 0.25 * rounds(m_tiles > 1.0 + chance ? m_tiles - chance : 1.0) + 0.5 * rounds(m_tiles) + 0.25 * rounds(m_tiles + chance);
        const double cost = (fourth(us) + fourth(memory) + fourth(m_tiles * units * (t.m + t.n) * K * 2.0 / from_caches)) * (f == base ? fourth(ahead) : 1.0);
        if (cost < best_cost) {
            best_cost = cost;
            best = f;
        }
    }
    return best;
}

}  // namespace paras
