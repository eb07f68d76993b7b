// spike_rules.h -- choices that depend on a system's sizes and the device alone (so a system gets the same bits
// alone and in a batch): plain C++, so that a host compiler builds them too (the tests hold them against
// measured times of both sides).
#pragma once
#include <cstdint>

// Residual kernel of a real system (block size 16 nt, nnz entries, m columns of the chunk): true for
// k_residual_mm (dense 16-row tiles), false for k_residual (gather).  The choice follows from the system and
// its columns in the chunk alone (a system gets the same bits alone and in a batch).  The gather kernel's time
// follows the entries per row and the columns; the dense tile's hardly depends on the entries, but on the
// tile's width w and on the occupancy its LDS leaves, so on nt.  us per residual, gather / dense tile:
//   k = 2, 10^6 rows: 1 column 59 / 60, 8 columns 78 / 71, 16 columns 175 / 96
//   k = 16, 600000 rows, 1 column: 5% fill 36 / 41, 20% 48 / 45; 16 columns: 2% fill 106 / 58
//   k = 24, 500000 rows, 1 column: 20% fill 48 / 61, 60% 88 / 74; 16 columns: 2% fill 86 / 68
//   k = 64, 300000 rows: 2% fill (3.6 entries per row), 16 columns 57 / 69, 64 columns 198 / 182; 5%, 16 columns 63 / 72
//   k = 64: 8 columns, 20% fill 66 / 81, 35% 110 / 96; 16 columns, 10% 76 / 79, 20% 98 / 85; 32 columns, 10% 135 / 116
//   k = 128, 200000 rows: 64 columns, 5% fill 201 / 252, 10% 270 / 255, 20% 380 / 280; 32 columns, 20% 202 / 188
// The lines below are where the two meet over k = 1..128, one-sided and unequal bands, fills of 2% to 100% and
// 1 to 64 columns.  Up to 16 columns b = 128 keeps the gather kernel (its tile leaves one workgroup per CU; it
// would win from about half the band filled: k = 128, full band, 16 columns 371 / 300).
inline bool dense_tile_residual(int nt, int n, int64_t nnz, int ku, int kl, int m) {
    const double nz = (double)nnz / n, w = ku + kl + 1.0;
    switch (nt) {
    case 1: return m > 8 || nz + 0.5 * m >= 5.7;
    case 2: return m > 8 || nz + 0.5 * m >= 13.5 + w / 6;
    case 4: return m > 32 || nz >= (m > 16 ? (w - 80) / 6 : (m > 8 ? w / 7 : 27 + w / 4 - 2 * m));
    case 8: return m > 32 ? nz >= 0.12 * w : m > 16 && nz >= 0.25 * w;
    default: return false;                      // b = 256: the tile does not fit the LDS
    }
}

// Band LU of one system: true for k_gbtrf_blk (panels), false for k_gbtrf (column by column).  Real bands take
// the panels wherever their LDS holds the multipliers.  Complex panels are half as wide and pay more per row of
// kl, so narrow bands and those with few superdiagonals stay with the columns.  us for 1000 columns, columns /
// panels, complex (kl, ku): (1, 1) 1950 / 3360, (64, 64) 3472 / 4013, (90, 90) 4618 / 4556, (100, 100) 5114 / 4942,
// (200, 200) 12598 / 7113, (60, 200) 5192 / 4665, (200, 60) 5572 / 6416, (400, 5) 7705 / 10422, (30, 448) 5400 / 4495;
// real: (1, 1) 1597 / 1271, (100, 100) 4557 / 1844, (400, 5) 11318 / 3235.
constexpr int BAND_PANEL_KL_MAX = 448;
inline bool band_lu_panels(bool cplx, int kl, int ku) {
    if (kl > BAND_PANEL_KL_MAX) return false;
    return !cplx || 3e-4 * kl * ku >= 1.6 + 0.01 * kl + 0.003 * ku;
}

// Partition count where the device's factor workgroups (`slots`) cap it.  Every partition has n / P rows and the
// last one the remainder too, up to P - 1 rows: with thousands of short partitions that is a chain many times
// the others' (10^6 rows on 3072 partitions: 121 blocks of 16 rows behind 3071 chains of 21; one column 424 us per
// FP64 solve, 285 on 3584 partitions, whose last chain has 22).  If the remainder exceeds a partition, the count up
// to a tenth below with the shortest last chain is taken.
inline long capped_partitions(long n, long slots, int b) {
    auto last_chain = [&](long p) { return (n - (p - 1) * (n / p) + b - 1) / b; };
    if (slots < 1 || n - slots * (n / slots) <= n / slots) return slots;
    long best = slots;
    for (long p = slots - 1; p >= slots - slots / 10; --p)
        if (last_chain(p) < last_chain(best)) best = p;
    return best;
}
