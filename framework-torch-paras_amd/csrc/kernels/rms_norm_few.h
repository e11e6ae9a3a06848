// Which RMSNorm backward passes are one launch, rms_norm_bwd_few (host code, no HIP).
#pragma once

#include <cstdint>

namespace paras {

constexpr long kFewMax = 16384;          // elements of a row

// Up to how many rows dx and the column sums are one launch (rms_norm_bwd_few): where that stops being faster than the kernels that
// read g and x once.  us, those kernels and this one (bf16): 64 columns 787 rows 5.4 and 5.3, 1500 5.9 and 8.1; 512 columns 1500 rows 8.8 and
// 8.3, 3000 9.8 and 15.6; 1024 columns 33 rows 10.8 and 3.2, 1500 15.2 and 10.0, 2500 16.0 and 15.2; 4096 columns 77 rows 16.5 and 3.4, 2000
// 20.1 and 16.8; 8192 columns 2000 rows 31.6 and 30.2, 2500 32.6 and 39.7; 14656 columns 184 rows 62.2 and 9.8.  Rows that are not whole vectors:
// bf16 257 columns 1500 rows 9.6 and 9.8; 4001 columns 2000 rows 29.8 and 22.6; fp32 777 columns 1500 rows 14.1 and 12.9, 2000 15.4 and 15.7.
// Where the other way is three kernels at any size (fp64; fp32 beyond 8192 columns), whole vectors: fp32 5500 x 12160 357 and 253, fp64
// 5500 x 1000 49 and 43, 5500 x 4096 205 and 177.
inline long few_rows(int elem_size, bool whole, long H) {
    const bool k16 = elem_size == 2, k64 = elem_size == 8;
    if (!whole)            return H <= 700 || k64 ? 1000 : k16 ? 2000 : 1500;
    if (k16)               return H <= 128 ? 700 : H <= 512 ? 1500 : 2000;
    return k64 || H > 8192 ? 5500 : 2000;
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
