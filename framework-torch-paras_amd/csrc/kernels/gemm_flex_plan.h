// Which tiles a 16-bit product runs on, and in how many parts of the contraction (host code, no HIP).
#pragma once

#include <utility>

namespace paras {
namespace flex {

constexpr int kPlanStep = 64;        // contraction steps of a tile
constexpr int kTile128x128 = 4;      // the index of its two-stage form in the tile table
struct Plan {
    int  tile = 0;              // index into the tile table
    int  splits = 1;            // parts of the contraction
    long k_per_split = 0;
};

// Per tile form: rows, columns, stages, workgroups a CU holds at once, and what a fit makes of one tile of 64
// contraction steps, in us: on a CU that is full (`step`), and at least, on a CU with fewer workgroups (`lat`: a
// barrier and the way from L2).  Coefficients of the estimate below, whose sum was fitted and counts; each by itself is no time or rate of the chip.
struct Tile { int m, n, stages, per_cu; double step, lat; };
constexpr Tile kTiles[] = {{256, 256, 2, 1, 0.827, 0.304}, {192, 256, 2, 1, 0.743, 0.052}, {192, 192, 3, 1, 0.682, 0.258}, {192, 128, 4, 1, 0.525, 0.562},
                           {128, 128, 2, 2, 0.849, 0.859}, {128, 128, 4, 1, 0.399, 0.472}, {64, 128, 2, 3, 0.916, 0.653}, {64, 128, 4, 1, 0.338, 0.230},
                           {64, 64, 3, 3, 0.753, 0.057},   {64, 64, 4, 2, 0.425, 0.147},   {128, 64, 3, 2, 0.677, 0.381}, {32, 64, 4, 3, 0.516, 0.183},
                           {192, 128, 2, 2, 1.439, 0.400}, {96, 128, 4, 1, 0.212, 0.413},  {96, 128, 2, 2, 0.655, 0.682}, {96, 64, 4, 2, 0.578, 0.279},
                           {160, 128, 2, 2, 1.460, 0.262}, {256, 224, 2, 1, 0.769, 0.527}, {192, 224, 2, 1, 0.735, 0.296}};
// From kFirstOddRows on the rows are an odd multiple of 32, which A cannot have where it lies along its rows; the last two are for both operands
// along the contraction only.  They come in whole rounds of workgroups, or fill the CUs, where the others do not: 1500 x 14336 x 4096 in bf16
// 448 tiles of 192 x 256 in two rounds 150 us, 512 of 192 x 224 146; 96 x 64 with four stages, two to a CU, 1136 x 1024 x 3584 20.2 (64 x 128) -> 17.8,
// 344 x 3584 x 1024 9.5 -> 8.8, 72 x 14336 x 4096 31.7 -> 29.6; 96 x 128 582 x 3584 x 1024 13.5 (128 x 128) -> 11.4, 1167 x 2048 x 2048 19.4 -> 16.9.  192 x 128
// two to a CU hides a tile's stores behind the other's loads: 25 rows of gradient into 7936 x 1152 12.3 -> 10.8.  32 x 64: 512 x 896 x 489 6.3 -> 5.9.
constexpr int kFirstOddRows = 13, kAlongContraction = 17;
constexpr int kTileCount = sizeof(kTiles) / sizeof(kTiles[0]);
constexpr int kCus = 256;

// The least estimated time over tile forms and numbers of parts.  Rounds of workgroups times the time of
// their share of the contraction and of their stores, plus the second kernel where the contraction is in
// parts.  The constants were fitted to 55000 timings of 1620 problems (25 to 8192 rows, 64 to 14336 columns, contractions of
// 25 to 14336, all three layouts, operands and weights from HBM): over them the choice is 0.7 % slower than the best form measured in the mean and
// 4.6 % at the 95th percentile (before the 96-row, 32 x 64 and two-to-a-CU forms 4.8 % and 15.6 %).  What the rule trades: a 256 x 256 tile reads half
// as much per flop as a 128 x 128 one, but with 192 of them for 256 CUs a quarter of the chip idles (3000 x 4096 x 4096 85.7 us, with 256 tiles of
// 192 x 256 78.3); a small problem has few workgroups per CU, and then more
// stages stand in for the other workgroups' loads (821 x 1024 x 3584 64 x 64: two stages in four parts 21 us, four stages 14.5 whole);
// what is still too few tiles is cut up along the contraction (1500 x 4096 x 14336, with the second
// kernel: 192 x 256 in two parts 141 us, 256 x 224 159; 192 x 128 whole 164).
//
// The search is on the way of every call, and a small product's launch costs a few us: the forms' constants are the compiler's
// (no division by a variable but two per number of parts), and forms and numbers of parts are left out whose least possible time is no
// better than one found.  The same plan as the search through all of them; host time of that and of this: 48 x 1024 x 1024 0.50 and 0.18 us,
// 128 x 2048 x 2048 0.68 and 0.36, 1024 x 1024 x 4096 0.67 and 0.25, 8192^3 0.15 and 0.08; 900 problems of 33 to 8192 rows 0.20 in the mean.
struct Search {
    int M, N, batch, k_tiles;
    bool may_split;
    double mn, memory;                          // elements of the result; us for the operands' way from memory
    double k_step, k_lat;                       // the layout's share in the forms' times
    int per[9], parts[9];                       // of the contraction, for 1, 2, 3, 4, 6, 9, 13, 19, 28 parts wanted
    int known = 0;
    double best_us = 1e30, found = 1e30;        // of `best`; of any form looked at
    Plan best;

    void want(int i, int wanted) {
        if (i < known) return;
        per[i] = static_cast<unsigned>(k_tiles + wanted - 1) / static_cast<unsigned>(wanted);
        parts[i] = static_cast<unsigned>(k_tiles + per[i] - 1) / static_cast<unsigned>(per[i]);
        known = i + 1;
    }
    template <int t, bool record> void consider() {
        constexpr Tile tl = kTiles[t];
        if (tl.m >= 128 && M <= 64 && batch == 1 && k_tiles <= 256) return;       // (half as many rows: not behind)
        constexpr int slots = kCus * tl.per_cu;
        constexpr double area = tl.m * tl.n / 65536.0, whole = area * (tl.per_cu > 1 ? 0.475 : 1.0) * 10.06, in_parts = area * (tl.per_cu > 1 ? 0.475 : 1.0) * 5.67;
        const double each = tl.step / tl.per_cu * k_step, lat = tl.lat * k_lat;
        const int tiles = (static_cast<unsigned>(M) + (tl.m - 1)) / tl.m * ((static_cast<unsigned>(N) + (tl.n - 1)) / tl.n) * batch;     // below 2^25
        // no less than the CUs' arithmetic and stores, shared out evenly, take
        const double least = (kStart + tiles * (k_tiles * each + whole) / kCus) * kBelow;
        if (least >= found) return;
        for (int i = 0, wanted = 1; wanted <= (may_split ? 32 : 1); ++i, wanted = wanted < 4 ? wanted + 1 : wanted + wanted / 2) {
            if (wanted > 1 && (wanted * 2 > k_tiles || tiles * wanted > 1600)) break;
            want(i, wanted);
            const int n_parts = parts[i], turns = static_cast<unsigned>(per[i] + (tl.stages - 1)) / tl.stages * tl.stages;
            const double finish = n_parts > 1 ? 2.5 + mn * n_parts * 1.574e-6 : 0.0;
            const double stores = n_parts > 1 ? in_parts : whole;
            if (least + finish >= found || (kStart + in_parts) * kBelow + finish >= found) break;       // (more parts are more to add)
            if ((turns * (each > lat ? each : lat) + kStart + stores) * kBelow + finish >= found) continue;      // a workgroup's own time
            const int wgs = tiles * n_parts, full = static_cast<unsigned>(wgs) / slots;
            const int rest = static_cast<unsigned>(wgs - full * slots + kCus - 1) / kCus;
            auto round = [&](double n) {
                const double c = each * n;
                return turns * (c > lat ? c : lat) + kStart + stores * n;
            };
            double us = full * round(tl.per_cu) + (rest > 0 ? round(rest) : 0.0);
            if (us < memory) us = memory;
            us += finish;
            if (us * kAbove < found) found = us * kAbove;
            if (record && us < best_us) {
                best_us = us;
                best.tile = t;
                best.splits = n_parts;
                best.k_per_split = static_cast<long>(per[i]) * kPlanStep;
            }
        }
    }
    template <int... t> void consider_all(std::integer_sequence<int, t...>, bool large, int forms) {
        consider<kUsual, false>();              // (so that the others have something to be measured against)
        // (best_us <= memory: nothing is better)
        (void)((best_us <= memory ||
                (t < forms && (kTiles[t].m * kTiles[t].n <= 128 * 128 || kTiles[t].per_cu > 1 || large) ? consider<t, true>() : void(), false)) || ...);
    }
    static constexpr int kUsual = 9;                                        // 64 x 64, four stages: a quarter of all choices
    static constexpr double kStart = 2.99;
    static constexpr double kBelow = 1.0 - 1e-9, kAbove = 1.0 + 1e-9;       // the bounds are other sums than the estimate
};

// Operands either way round: `a_rows`, `b_rows` as in Problem (sizes as takes() has them: M and N below 2^31, batch below 2^16).
inline Plan plan_of(long M, long N, long K, long batch, bool a_rows, bool b_rows, bool may_split) {
    Search s;
    s.M = static_cast<int>(M); s.N = static_cast<int>(N); s.batch = static_cast<int>(batch);       // (takes(): below 2^30, 2^31 and 2^16)
    s.k_tiles = static_cast<int>((K + kPlanStep - 1) / kPlanStep);
    s.may_split = may_split;
    s.mn = static_cast<double>(M) * N * batch;
    s.memory = static_cast<double>(M + N) * K * batch * 2 / 10.86e6 + 3.75;
    s.k_step = a_rows ? 1.069 : b_rows ? 1.222 : 1.0;
    s.k_lat = b_rows && !a_rows ? 1.084 : 1.0;
    // (K <= 512: mostly stores, and tiles of which a CU holds several overlap them with other tiles' work)
    s.consider_all(std::make_integer_sequence<int, kTileCount>{}, K > 512, a_rows ? kFirstOddRows : b_rows ? kAlongContraction : kTileCount);
    return s.best;
}

}  // namespace flex
}  // namespace paras
