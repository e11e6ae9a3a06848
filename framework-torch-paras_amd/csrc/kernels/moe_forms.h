// Which tiles a grouped product of an expert layer runs on (host code, no HIP).
#pragma once

#include <cmath>
#include <utility>

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

// All tiles of the grouped products: those above in their order, then what grouped_tile_kernel has besides.  (A time of zero: not for that product.)  The
// times are of grouped_tiles' fit.
inline constexpr GroupedForm kAllForms[] = {{128, 128, 2, 2, {1.270, 1.004}, {0.980, 0.773}}, {128, 128, 3, 1, {0.615, 0.497}, {0.381, 0.529}},
                                             {64, 128, 2, 3, {1.380, 1.153}, {0.789, 0.673}}, {64, 128, 4, 1, {0.228, 0.208}, {0.499, 0.412}},
                                             {32, 128, 4, 2, {0.919, 0.726}, {0.104, 0.287}}, {256, 256, 2, 1, {1.516, 1.166}, {0.251, 0.266}},
                                             {256, 256, 2, 1, {1.228, 1.068}, {0.261, 0.319}}, {32, 64, 4, 3, {0.583, 0.552}, {0.186, 0.245}},
                                             {64, 64, 4, 2, {0.579, 0.506}, {0.340, 0.297}}, {96, 64, 4, 2, {0.676, 0.589}, {0.351, 0.319}},
                                             {96, 128, 2, 2, {1.187, 0.897}, {0.772, 0.763}}, {192, 128, 2, 2, {1.513, 1.217}, {0.903, 0.858}},
                                             {160, 128, 2, 2, {1.358, 0.000}, {0.918, 0.000}}, {192, 256, 2, 1, {0.000, 0.990}, {0.000, 0.162}},
                                             {128, 256, 3, 1, {0.000, 0.832}, {0.000, 0.476}}};
constexpr int kAllFormCount = sizeof(kAllForms) / sizeof(kAllForms[0]);

// Tiles of m rows where each of E experts has R / E rows on average and each row is sent on its own (a normal distribution): the number to be expected and its standard
// deviation.  An expert has a tile more for each multiple of m that its rows exceed; where it fills more than six, half a tile is what is lost.  (The normal
// distribution's tail as the logistic function of 1.5976 z + 0.07056 z^3, Bowling et al. 2009: within 2e-4.)
inline void tiles_of_rows(long E, long R, int m, double* tiles, double* spread) {
    const double rows = static_cast<double>(R) / E;
    if (rows > 6.0 * m) {
        *tiles = E * (rows / m + 0.5);
        *spread = std::sqrt(E / 12.0);
        return;
    }
    const double per = 1.0 / std::sqrt(rows);
    double more = 1.0 - std::exp(-rows), n = more, var = more * (1.0 - more), fewer = 1.0 - more;          // P(a tile more), and of all up to here the sums
    for (double j = m; (j - rows) * per < 4.25; j += m) {
        const double z = (j + 0.5 - rows) * per;
        more = 1.0 / (1.0 + std::exp(z * (1.5976 + 0.07056 * z * z)));
        n += more;
        var += more * (1.0 - more + 2.0 * fewer);
        fewer += 1.0 - more;
    }
    *tiles = E * n;
    *spread = std::sqrt(E * var);
}

// The tiles that a product runs on.  grouped_form's choice stays unless another form is estimated to be 7 % (gate-up) or 5 % (down) faster, by three times that overlap for the most
// part (the fourth root of the sum of their fourth powers): rounds of workgroups, each of its contraction, start and stores; the way of the weights from memory; that of all
// tiles' operands from the caches.
//   The number of an expert's tiles is a matter of chance, and one tile more can be a round more: grouped_form's choice is estimated half with the expected number and half with
// 1.2 standard deviations fewer, every other with as many more.  Gate-up of 3221 tokens, top-2, 8 experts, 1088 x 832 expects 511 tiles of 192 x 128 for 512 places, and came to
// 520 (layer 75 -> 93 us): it stays on 256 x 256.  So do 1956 tokens, 896 x 8000, where 192 x 128 is 260 -> 241 us in seven of eight routings, and 249 -> 293 in the one whose experts'
// 256-row tiles are 16 and not 17.
//   Fitted to 59000 timings of 2212 layers (4 to 64 experts, 8 to 49152 routed rows, H 512 to 4096, I 512 to 14336, weights from HBM), no tile faster than the matrix cores' 2.5
// PFLOP/s, no more than 8 TB/s from memory and 40 from the caches.  Of 400 layers that the fit
// has not seen 8.4 % faster in the mean than with grouped_form's choices, 270 of them more than 3 %, four 5 to 8 % slower.
// Beyond 128 experts, 65536 rows and sizes of 16384 grouped_form chooses alone.  A form that cannot be as fast by its contraction shared out over all CUs is not looked at any
// further: 0.2 to 0.75 us of host time for a choice, of which grouped_form 0.10 to 0.17.
//   What the further forms bring.  32 x 64 with four stages, three to a CU, is for
// products whose tiles are too few for 256 CUs: down of 230 tokens, top-2, 8 experts, 640 x 4096, 26.8 us on 32 x 128, 19.5.  192 x 128 and 160 x 128 with two stages,
// two to a CU, hide each other's SwiGLU and stores, which 256 x 256 tiles do one CU at a time, and waste less of an expert's last tile: gate-up of 2167 tokens,
// top-4, 32 experts, 1856 x 1280, 181 us on 256 x 256, 166.  192 x 256 and 128 x 256: down of 1156 tokens, top-2, 8 experts, 3520 x 14272, and of 910,
// 3008 x 10496 (with the gate-up product's change layers 1201 -> 860 and 596 -> 467).
template <bool kSwiglu> struct TileChoice {
    static constexpr int w = kSwiglu ? 0 : 1;
    static constexpr double start = kSwiglu ? 0.748 : 0.000, store = kSwiglu ? 31.197 : 4.357;          // us
    static constexpr double supers = kSwiglu ? 0.979 : 1.199, one_by_one = kSwiglu ? 0.999 : 1.165;          // grouped_gemm_direct_kernel's starts and stores, against the others'
    static constexpr double from_memory = kSwiglu ? 5.88e6 : 7.87e6, from_caches = kSwiglu ? 35.6e6 : 40.0e6;          // bytes per us
    static constexpr double kDoubt = 1.2;
    long E, R, N, K;
    int base, best;
    double rounds_256;                // of 256 x 256 tiles
    double ahead, used, memory, best_us, best_cost;
    double by_rows[9][2];             // row tiles of 32, 64 ... 256, and their spread

    static double fourth(double v) { return v * v * v * v; }
    static double root(double v) { return std::sqrt(std::sqrt(v)); }
    static double larger(double a, double b) { return a > b ? a : b; }
    static double down(double v) { return static_cast<double>(static_cast<long>(v)); }          // (of what is not negative; std::floor and std::ceil are calls)
    static double up(double v) { return down(v) + (down(v) < v); }
    template <int f> void consider() {
        constexpr GroupedForm t = kAllForms[f];
        constexpr long cols = kSwiglu ? t.n / 2 : t.n;
        constexpr double ends = f == kDirectForm ? supers : f == kOneByOne ? one_by_one : 1.0, each = t.step[w] / t.per_cu, lat = t.lat[w];
        constexpr double begin = start * ends, stores = store * ends * t.m * cols / 65536.0, slots = 256.0 * t.per_cu;
        const unsigned n_units = static_cast<unsigned>(N + cols - 1) / static_cast<unsigned>(cols), k_tiles = static_cast<unsigned>(K + kFormStep - 1) / kFormStep;
        const double units = n_units, turns = (k_tiles + t.stages - 1) / t.stages * t.stages, traffic = units * (t.m + t.n) * K * (2.0 / from_caches);
        if (f != base) {
            const double least_tiles = larger(R * (1.0 / t.m), used);
            const double least = larger(least_tiles * units * (turns * each + (t.per_cu > 1 ? 0.0 : stores)) / 256.0, turns * larger(each, lat) + stores) + begin;
            if (fourth(least) + memory + fourth(least_tiles * traffic) >= best_cost) return;
        }
        double* const tiles = by_rows[t.m / 32];
        if (tiles[0] == 0.0) tiles_of_rows(E, R, t.m, &tiles[0], &tiles[1]);
        // n workgroups on a CU: several hide their stores (and SwiGLU) behind each other's contraction as far as either is longer
        auto round = [&](double n) {
            const double loop = turns * larger(each * n, lat), out = stores * n;
            if (n < 2) return begin + loop + out;
            return begin + (kSwiglu ? std::sqrt(loop * loop + out * out) : root(fourth(loop) + fourth(out)));
        };
        auto rounds = [&](double m) {
            if (f == kDirectForm) return up(m / kSuperM * up(units / kSuperN) / 8) * round(1);
            if (f == kOneByOne) return up(m * units / 256) * round(1);
            const double full = down(m * units / slots), rest = up((m * units - full * slots) / 256);
            return full * round(t.per_cu) + (rest > 0 ? round(rest) : 0.0);
        };
        const double others = memory + fourth(tiles[0] * traffic), expected = fourth(rounds(tiles[0])) + others;
        const double doubt = fourth(rounds(f == base ? larger(tiles[0] - kDoubt * tiles[1], 1.0) : tiles[0] + kDoubt * tiles[1])) + others;
        const double us = (f == base ? ahead : 1.0) * (root(expected) + root(doubt));
        if (f == base || us < best_us) {
            best_us = us;
            best_cost = fourth(0.5 * us);
            best = f;
        }
    }
    template <int... f> void consider_all(std::integer_sequence<int, f...>) {
        ((f == base ? consider<f>() : void()), ...);
        // (256 x 256 tiles: from 40 rows an expert, where they were timed.  One by one: gate-up of up to twenty rounds, beyond which the two are level; of down one round too many is a
        // long one, and grouped_form's word counts)
        auto may = [&](int g) { return (g != kDirectForm && g != kOneByOne) || (R >= 40 * E && rounds_256 <= 20 && (g == kDirectForm || kSwiglu)); };
        ((f != base && kAllForms[f].step[w] > 0.0 && may(f) ? consider<f>() : void()), ...);
    }
};
template <bool kSwiglu> int tile_choice(long E, long R, long N, long K, int base) {
    constexpr long cols = kSwiglu ? 128 : 256;
    const double rounds_256 = static_cast<double>(R) / 256 * ((N + cols - 1) / cols) / 256;
    const int as = base == kDirectForm && rounds_256 > 20 ? kOneByOne : base;         // (super-tiles are estimated in whole ones, which of few rounds is right)
    // (gate-up with many super-tiles over a short contraction: what the estimate gives the smaller tiles for hiding each other's SwiGLU is too much there)
    const double ahead = !kSwiglu ? 0.95 : base == kDirectForm && K <= 1024 && rounds_256 > 3 ? 0.85 : 0.93;
    TileChoice<kSwiglu> c{E, R, N, K, as, as, rounds_256, ahead, static_cast<double>(R < E ? R : E), 0.0, 0.0, 0.0, {}};
    c.memory = c.fourth(c.used * N * K * ((kSwiglu ? 4.0 : 2.0) / c.from_memory));
    c.consider_all(std::make_integer_sequence<int, kAllFormCount>{});
    return c.best == as ? base : c.best;
}
inline int grouped_tiles(bool swiglu, long E, long R, long N, long K) {
    const int base = grouped_form(swiglu, E, R, N, K);
    if (E > 128 || R > 65536 || N > 16384 || K > 16384) return base;
    return swiglu ? tile_choice<true>(E, R, N, K, base) : tile_choice<false>(E, R, N, K, base);
}

}  // namespace paras
