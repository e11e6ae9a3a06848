// Which form of sdpa_f32_kernel a problem runs on (host code, no HIP).
#pragma once

#include "paras_hip.h"

namespace paras {

// Queries by keys of a turn in the fp32 form.  Turns of 16 keys for 16 queries take the fewest registers, and what they leave room for, two workgroups per CU at 128
// elements and four at 64, is worth more than the operands that larger blocks share, but not everywhere.  The figures are us of 16 x 16 / 16 x 32 / 32 x 32 keys, from 90
// problems, each without a mask, causal, with 30 % of the keys padded and with an additive mask, with the weights returned and without.
//   Whether weights are returned changes the queries of a block at most, and not the keys of a turn, so the output is the same bits either way.
enum class Form { k16x16, k32x16, k16x32, k32x32 };
template <int DM>
Form form_of(const paras_sdpa_args& a) {
    const long heads = a.B * a.Hq, blocks = (a.Lq + 15) / 16 * heads, pairs = (a.Lq + 31) / 32 * heads;
    const bool causal = a.is_causal != 0, padded = a.mask_kind == 1, added = a.mask_kind == 2;
    const double scores = static_cast<double>(heads) * static_cast<double>(a.Lq) * static_cast<double>(a.Lk);
    if (DM == 64) {
        // Four workgroups of 16 x 16 per CU are ahead up to a few turns each; beyond, turns of 32 keys wait for half as many row maxima (B1 H4 S4000 causal 192 /
        // 150 / 184, B1 H1 S3000 49 / 47 / 81).  Blocks of 32 queries, two per CU, where they come in whole rounds: unmasked B2 H16 S2048 397 / 398 / 382; with an
        // additive mask, B2 H16 S2048 519 / 531 / 449, B1 H8 S2048 (one round) 137 / 137 / 125, B1 H64 S600 106 / 111 / 100; between whole rounds B1 H16
        // S1500 134 / 141 / 135, B2 H16 S600 57 / 59 / 64.
        if (a.Lk <= 320) return Form::k16x16;
        if (added && (pairs >= 1000 || (pairs >= 448 && pairs <= 512 && a.Lk >= 1000))) return Form::k32x32;
        if (added && pairs > 512 && a.Lk <= 2000) return Form::k16x16;
        if (!padded && !added && !causal && pairs >= 448) return Form::k32x32;
        if (causal && pairs >= 448 && a.Lk <= 640) return Form::k16x16;              // (B8 H16 S512 109 / 113 / 109)
        return Form::k16x32;
    }
    if (DM == 128) {
        // Two workgroups of 16 x 16 per CU: B2 H16 S2048 695 / 833 / 746, B1 H64 S300 46 / 70 / 73, B3 H8 S145 causal 10 / 12 / 21.  One per CU and larger turns
        // where there is no second one for most CUs: masks, B1 H1 S3000 padded 85 / 82 / 136, additive 95 / 84 / 162; causal, where the second ones are the
        // longest tiles of the next head, on the CUs that have the longest of the first: B1 H2 S3000 112 / 80 / 134, S4096 175 / 131 / 177, B1 H1 S8192 274 / 240 / 345 (but
        // S8256, 516 blocks, 274 / 289 / 350), B1 H3 S2000 88 / 72 / 93, B2 H2 S1100 39 / 33 / 56 (but B1 H3 S2500, 471 blocks, 97 / 105 / 115; B1 H5 S1200 49 / 52 / 61).
        // Blocks of 32 queries for long causal rows where they just fill the CUs once or twice over: B1 H2 S6144 282 / 291 / 264, S7680 444 / 432 / 374, S8192 487 / 481 /
        // 432, S8256 491 / 530 / 494, B1 H4 S7168 680 / 765 / 692, S8192 885 / 961 / 862, B1 H1 S16384 833 / 930 / 813.
        if ((padded || added) && blocks <= 256 && a.Lk >= (added ? 900 : 1200)) return Form::k16x32;
        if (causal && blocks > 256 && (blocks <= 300 || (blocks <= 448 && heads == 3) || (blocks <= 512 && heads <= 2)) && a.Lk >= 900) return Form::k16x32;
        if (causal && a.Lk >= 6000 && ((pairs >= (heads == 1 ? 490 : 380) && pairs <= 512) || (pairs >= 950 && pairs <= 1024))) return Form::k32x32;
        // 32 queries by 16 keys read K and V half as often, in the registers of two workgroups per CU still.  Where more weights are written than the last-level cache holds
        // (16 x 16 / 32 x 16 / 32 x 32: B2 H16 S2048 unmasked 990 / 925 / 981, padded 1051 / 950 / 1021, additive 1103 / 998 / 1067; B1 H8 S4096 995 / 926 / 961, 1064 /
        // 960 / 993, 1111 / 999 / 1042; but B1 H7 S4000, 875 pairs, 815 / 855: over one to a CU and not two in the last round), and for long rows of an additive
        // mask (B1 H8 S4096 818 / 730 / 793, B1 H2 S8192 831 / 731 / 806).
        const bool ragged = pairs < 1536 && pairs % 512 > 256 && pairs % 512 < 448;
        if (a.attn != nullptr && !causal && scores >= 96e6 && !ragged) return Form::k32x16;
        if (added && a.Lk >= 4096) return Form::k32x16;
        return Form::k16x16;
    }
    // 256 elements, one workgroup per CU: 16 x 16 leaves the registers for what is requested ahead, 16 x 32 waits for half as many row maxima, which counts over
    // many turns, and reads and writes rows of weights in longer pieces: B2 H16 S600 179 / 188, S2048 1629 / 1609, with the weights 2010 / 1838, B4 H16 S2048
    // 3463 / 3215, B1 H1 S5000 484 / 463; B1 H32 S1500 931 / 931, with the weights 1119 / 1055.  Up to 80 keys one wave would take a second turn of 16 for the
    // last of them, up to 96 more or less (B9 H16 S66 37 / 35, additive 39 / 36, B7 H8 S86 26.0 / 25.5; a mask or the causal rule may close that one: 35 / 38 padded).
    if (a.Lk >= (causal ? 4000 : 2000) || (!causal && scores >= 64e6) || (a.Lk > 64 && a.Lk <= 96 && !causal && !padded)) return Form::k16x32;
    return Form::k16x16;
}

}  // namespace paras
