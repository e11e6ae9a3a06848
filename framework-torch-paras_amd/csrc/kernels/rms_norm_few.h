// Which RMSNorm backward passes are one launch, rms_norm_bwd_few (host code, no HIP).
#pragma once

#include <cstdint>

namespace paras {

constexpr long kFewMax = 16384;          // elements of a row

// Up to how many rows dx and the column sums are one launch (rms_norm_bwd_few): where that stops being faster than the kernels that
// read g and x once, by 2200 pairs of timings.  A column workgroup's time grows with the rows; where the last one has a single 16-byte piece of each row (or up to four
// elements, of rows that are not whole pieces) its lines are fetched for little and it takes half as long again.  us, those kernels and this one.  bf16: 64 columns
// 700 rows 5.3 and 5.3, 1000 5.4 and 6.2; 72 columns 400 5.3 and 4.2, 500 5.3 and 5.6; 136 columns 600 6.1 and 5.5, 700 6.2 and 6.7; 256 columns 1000 6.5 and 6.3, 1250 6.5 and 7.5;
// 392 columns 900 8.8 and 8.3, 1100 9.1 and 9.5; 488 columns 1250 9.5 and 9.6, 1500 9.6 and 10.8; 584 columns 1750 15.7 and 14.8, 2000 15.8 and 18.5; 1024 columns 33 rows 10.8 and 3.2,
// 2000 15.4 and 12.9; 4096 columns 77 rows 16.5 and 3.4, 2000 20.1 and 16.8; 8192 columns 2000 31.6 and 30.2, 2500 32.6 and 39.7; 14656 columns 184 rows 62.2 and 9.8.
// Rows that are not whole pieces: 65 columns 850 7.9 and 7.8, 1000 8.0 and 9.4; 385 columns 1000 9.1 and 8.1, 1250 10.0 and 10.2; 2001 columns 2000 22.4 and 15.4.
// fp32: 68 columns 1500 8.3 and 7.0, 2000 8.7 and 11.5; 132 columns 1250 8.4 and 7.2, 1500 8.7 and 9.1; 292 columns 1800 11.9 and 11.0, 2000 12.2 and 12.8; 1000 columns 2000 16.2 and 14.4;
// 33 columns 800 7.4 and 7.1, 1000 7.6 and 8.6; 777 columns 1500 14.0 and 12.8.  Where the other way is three kernels at any size (fp64; fp32 beyond 8192 columns), whole pieces:
// fp32 8196 columns 5500 rows 237 and 186; fp64 128 columns 2000 11.6 and 9.1, 2500 12.2 and 13.2; 130 columns 1500 10.5 and 9.9, 2000 11.7 and 12.6; 512 columns 3000 18.4 and 17.8,
// 3500 19.9 and 20.3; 642 columns 2000 17.5 and 16.5, 2500 19.2 and 19.9; 4096 columns 5500 205 and 177; not: 193 columns 500 7.9 and 7.1, 700 8.5 and 9.8; 769 columns 900 14.1 and 12.5,
// 1000 14.5 and 15.0.
inline long few_rows(int elem_size, bool whole, long H) {
    const bool k16 = elem_size == 2, k64 = elem_size == 8;
    if (!whole) {
        if (k64)      return H <= 256 ? 550 : H <= 384 ? 700 : H < 900 ? 900 : 1000;
        if (H <= 128) return H % 32 >= 1 && H % 32 <= 4 ? 800 : 1000;
        return H <= 700 ? 1000 : k16 ? 2000 : 1500;
    }
    const bool one_piece = H * elem_size % 128 == 16;
    if (k16) return H <= 128 ? (one_piece ? 450 : 700) : H <= 256 ? (one_piece ? 600 : 1000) : H <= 512 ? (one_piece ? 900 : 1250) : one_piece && H < 1024 ? 1750 : 2000;
    if (k64) return one_piece ? (H <= 256 ? 1500 : H < 1000 ? 2000 : 5500) : H <= 160 ? 2200 : H <= 608 ? 3000 : 5500;
    if (one_piece && H <= 512) return H <= 96 ? 1700 : H <= 224 ? 1350 : 1800;
    return H > 8192 ? 5500 : 2000;
}

// Whether the pass is that launch.  `whole`: rows of whole aligned 16-byte pieces.
inline bool takes_few(int elem_size, const void* go, const void* x, const void* w, const float* rstd, const void* gx, const void* gw, long rows, long H, bool* whole) {
    auto at = [](const void* p) { return reinterpret_cast<std::uintptr_t>(p); };
    *whole = H * elem_size % 16 == 0 && ((at(go) | at(x) | at(w) | at(gx)) & 15) == 0;
    if (H > kFewMax || rows > few_rows(elem_size, *whole, H)) return false;
    // (Its workgroups write dx and dw while others of the same launch still read g, x, w and rstd: neither may share memory with those, nor with the other.  Of the kernels
    // of the other way only a later launch writes dw, and a row's dx is written by who has read the row.)
    const std::uintptr_t row = static_cast<std::uintptr_t>(H) * elem_size, all = static_cast<std::uintptr_t>(rows) * row, stats = static_cast<std::uintptr_t>(rows) * sizeof(float);
    auto apart = [&](const void* p, std::uintptr_t n, const void* q, std::uintptr_t m) { return at(p) + n <= at(q) || at(q) + m <= at(p); };
    auto from_inputs = [&](const void* p, std::uintptr_t n) { return apart(p, n, go, all) && apart(p, n, x, all) && apart(p, n, w, row) && apart(p, n, rstd, stats); };
    return from_inputs(gx, all) && from_inputs(gw, row) && apart(gx, all, gw, row);
}

}  // namespace paras
