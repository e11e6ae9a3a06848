// How the query tiles of a causal problem are dealt to the workgroups of sdpa_flash.hip (heads_together) and to the persistent ones of
// sdpa_flash_wide.hip (deal_of).  Host code, no HIP.
//
// The items of a pool of workgroups (the chip, or an XCD where the heads are dealt to the XCDs) are numbered by groups of G heads, longest query
// tiles first within a group, and dealt in rounds of one item per workgroup, every other round in reverse order.  A few heads at a time
// keep their keys and values in the caches, many at a time come out even: a workgroup that comes to long tiles every time holds up the rest
// (bf16 D128 B5 H8 S6175, 25 tiles of 25 heads for 32 workgroups: one head at a time 1.4 times the share, 436 us, five 1.02, 355; B5 H14 S3840, 1050 items for
// 256: 2.0 times and 382 us, all 70 heads 1.03 and 256).
#pragma once

#include <initializer_list>

namespace paras {
namespace flash {

struct Deal {
    int    group = 1;      // heads that are gone through together
    double cost  = 1e30;   // of an even deal out of the caches
};

constexpr long kDealWgs = 512;

// What the workgroup with the most gets, in tiles of keys, of `heads` heads of nq query tiles (1 .. nq tiles of keys each) in groups of G; and about how many
// steps it takes to know.  Either by runs of items of one length, which add the same to a stretch of workgroups, or by workgroups: those whose places differ by whole
// groups get the same, but for the last round, which only some of them have.
inline long steps_by_runs(long heads, long nq, long wgs, long G) { return heads / G * nq + heads * nq / wgs; }
inline long steps_by_places(long heads, long nq, long wgs, long G) { return (2 * G * nq < wgs ? 2 * G * nq : wgs) * (heads * nq / wgs + 1); }
inline long most_by_runs(long heads, long nq, long wgs, long G) {
    long step[kDealWgs + 1] = {};
    for (long item = 0, at = 0, len = nq, left = G, back = 0, items = heads * nq; item < items;) {
        const long n = left < wgs - at ? left : wgs - at, first = back ? wgs - at - n : at;
        step[first] += len;
        step[first + n] -= len;
        item += n;
        at += n;
        left -= n;
        if (at == wgs) {                 // the next round, the other way
            at = 0;
            back ^= 1;
        }
        if (left == 0) {
            left = G;
            if (--len == 0) len = nq;
        }
    }
    long most = 0, load = 0;
    for (long w = 0; w < wgs; ++w) {
        load += step[w];
        if (load > most) most = load;
    }
    return most;
}
inline long most_by_places(long heads, long nq, long wgs, long G) {
    const unsigned span = static_cast<unsigned>(G * nq), group = static_cast<unsigned>(G), two = static_cast<unsigned>(2 * wgs % span);
    const long rounds = heads * nq / wgs, rest = heads * nq % wgs;
    long most = 0;
    auto look = [&](long place) {                            // of the workgroup that has this place in the last round
        const long w = rounds & 1 ? wgs - 1 - place : place;
        unsigned there = static_cast<unsigned>(w % span), back = static_cast<unsigned>((2 * wgs - 1 - w) % span);
        long load = 0;
        for (long r = 0; r < rounds + (place < rest); r += 2) {
            load += nq - there / group;
            if (r + 1 < rounds + (place < rest)) load += nq - back / group;
            there += two;
            there -= there >= span ? span : 0;
            back += two;
            back -= back >= span ? span : 0;
        }
        if (load > most) most = load;
    };
    for (long place = 0; place < wgs && place < span; ++place) look(place);
    for (long place = rest; place < wgs && place < rest + span; ++place)
        if (place >= span) look(place);
    return most;
}

// The time of a deal, of an even one's: as fitted to 68 problems of 1408 to 8192 queries, each with up to six groups.  About half of what a workgroup gets
// over its share shows (the others' CUs rest, and its own runs faster), and groups whose keys and values take more than 128 MB between them, half the
// last-level cache, cost up to a tenth (B9 H28 S4096: 2 heads 1013 us, 252 of 528 MB 1129; B48 H32 S1536: 1083 and 1255).
inline double deal_cost(double share, long most, double group_bytes) {
    const double beyond = (group_bytes - 128e6) / 256e6;
    return (0.45 + 0.55 * static_cast<double>(most) / share) * (1.0 + 0.1 * (beyond < 0 ? 0 : beyond > 1 ? 1 : beyond));
}

// BH heads in all, of nq query tiles each, and `head_bytes` of keys and values per query head; `blocks` workgroups on the chip.  Up to five groups are looked
// at, until one is within 4 % of the best there can be: one head (first where an XCD has its own heads: its 4 MB of L2 are worth 1 to 3 %), the two largest that
// fit the cache, the next above, and all; none that takes many steps, for a call waits for its deal
// (0.7 us in the mean of 1000 problems, 1.2 at most where the kernel takes less than 200, 3 at most; walking every item of every group took 10 to 60).  Of those
// 1000 the best of all groups is missed by 0.2 % in the mean, by over 2 % in one of 20, by 6 % at most.
inline Deal deal_of(long BH, long nq, long blocks, double head_bytes) {
    Deal d;
    const bool by_xcd = BH % 8 == 0 && blocks % 8 == 0;
    const long heads = by_xcd ? BH / 8 : BH, wgs = by_xcd ? blocks / 8 : blocks;
    if (wgs < 1 || wgs > kDealWgs) return d;
    const double bytes = by_xcd ? 8 * head_bytes : head_bytes, share = 0.5 * static_cast<double>(heads * nq) * static_cast<double>(nq + 1) / static_cast<double>(wgs);
    long fits = 1, smaller = 1, larger = heads;              // divisors of `heads`: the largest whose keys and values fit, and its neighbours
    auto sort_in = [&](long g) {
        if (g > 1 && static_cast<double>(g) * bytes > 128e6) {
            if (g < larger) larger = g;
        } else if (g > fits) {
            smaller = fits;
            fits = g;
        } else if (g > smaller && g < fits) {
            smaller = g;
        }
    };
    for (long g = 1; g * g <= heads; ++g)
        if (heads % g == 0) {
            sort_in(g);
            sort_in(heads / g);
        }
    const long order[5] = {by_xcd ? 1 : fits, by_xcd ? fits : smaller, by_xcd ? smaller : larger, by_xcd ? larger : 1, heads};
    for (int i = 0; i < 5 && d.cost > 1.04; ++i) {
        const long g = order[i], runs = steps_by_runs(heads, nq, wgs, g), places = steps_by_places(heads, nq, wgs, g);
        bool seen = false;
        for (int j = 0; j < i; ++j) seen = seen || order[j] == g;
        if (seen || (g != heads && (runs < places ? runs : places) > (i == 0 ? 1024 : 512))) continue;
        const long most = runs <= places ? most_by_runs(heads, nq, wgs, g) : most_by_places(heads, nq, wgs, g);
        const double cost = deal_cost(share, most, static_cast<double>(g) * bytes);
        if (cost < d.cost) d = {static_cast<int>(g), cost};
    }
    return d;
}

// The kernel of 32 queries per wavefront: an XCD has `heads` heads of nq query tiles of 128 and takes the longest tiles of so many of them first.  One or two heads at
// a time, the last heads' longest tiles start late; of too many, keys and values are fetched again for every tile.  Over 110 problems, by one or two heads / this
// way: D64 B4 H16 S2048 54.4 / 45.7 us, B8 H8 S1024 21.9 / 17.5, B5 H8 (one key head) S2072 47.7 / 35.2; D128 B2 H32 S700 22.3 / 20.1, B20 H64 S134 51.9 / 42.9; D256 B2 H32 S934
// 70.2 / 59.9; the mean of all 0.945, none over 3 % slower.
//   More heads come out even in the first rounds of workgroups (two to a CU, one at 256 elements) than in later ones, where their number counts as their bytes do
// (D128 B29 H24 S308, 261 tiles: 1 head 53.0, 3 53.9, 29, which have 4.4 MB, 61.1; B7 H64 S602: 2 heads 75.0, 8 77.2, 14 81.2, 56 92.5).  A group divides the heads; where they
// hardly divide, one half as large again will do (19 heads, D64 S1749: one 90.3, all 81.0).
inline long heads_together(long heads, long nq, long Lk, long D) {
    const bool   few = heads * nq <= (D == 64 ? 192 : D == 128 ? 144 : 96);
    const double megabytes = D == 64 || (D == 128 && few) ? 8.0 : D == 128 ? 2.0 : 4.0;
    const double fit = megabytes * 1048576.0 / (static_cast<double>(Lk) * static_cast<double>(D) * 4.0), many = (few ? 2048.0 : 1024.0) / static_cast<double>(D);
    const double most = fit < many ? fit : many;
    long at_most = 1, above = heads;                         // the largest divisor of `heads` up to `most` and the next
    for (long g = 1; g * g <= heads; ++g)
        if (heads % g == 0)
            for (const long d : {g, heads / g}) {
                if (static_cast<double>(d) <= most) at_most = d > at_most ? d : at_most;
                else                                above = d < above ? d : above;
            }
    if (at_most <= 2 && 2.0 * static_cast<double>(at_most) < most && static_cast<double>(above) <= (D == 64 ? 2.0 : 1.5) * most) at_most = above;
    return at_most == 1 && heads % 2 == 0 ? 2 : at_most;
}

}  // namespace flash
}  // namespace paras
