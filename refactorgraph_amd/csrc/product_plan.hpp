// What the kernels of MatMul and MatMulInteger are expected to take, and the choice between them: plain functions of
// sizes (no device, no HIP), so that the choice itself is tested on the CPU.  All times are microseconds; the figures are
// least squares over launches of every kernel that takes a call, at sizes drawn over the ranges named with them.
#pragma once

#include <cstddef>
#include <cstdint>

namespace rg {

// ---------------------------------------------------------------- F32
//
// Fitted over 2,500 products of 1 to 256 rows, k 64 to 8320, 16 to 50257 columns; over them the choice takes 0.06 % longer
// than the faster kernel of each call.

// mm_rows (B as [n, k]) and mm_rows_kn (B as [k, n]): passes of up to 32 rows, a workgroup per 16 columns.  A round is 256
// workgroups; passes of more than 16 rows go in whole rounds (one wavefront per SIMD).
struct F32Pass {
    double fixed, per_k, per_round, per_work;  // us; per round and 1000 of k; per round; per 256 workgroups and 1000 of k
};
inline double f32_rows_us(size_t m, size_t k, size_t n, size_t count, bool b_is_nk) {
    constexpr F32Pass nk[] = {{1.8, 1.8, 0.48, 0.83}, {2.0, 2.3, 0.98, 1.07}, {3.1, 2.8, 0.54, 0.91}, {0.7, 5.6, 2.8, 0}};
    constexpr F32Pass kn[] = {{1.8, 0.85, 0.26, 2.8}, {1.5, 1.25, 0.8, 3.15}, {1.7, 1.7, 1.5, 3.6}, {0, 6.1, 4.1, 0}};
    const uint64_t workgroups = static_cast<uint64_t>((n + 15) / 16) * count;
    const double kilo = 1e-3 * static_cast<double>(k), work = static_cast<double>(workgroups) / 256;
    const double whole = static_cast<double>((workgroups + 255) / 256);
    auto pass = [&](size_t rows) -> double {
        const int i = rows <= 4 ? 0 : rows <= 8 ? 1 : rows <= 16 ? 2 : 3;
        const F32Pass &p = b_is_nk ? nk[i] : kn[i];
        return p.fixed + (i == 3 ? whole : work > 1 ? work : 1) * (p.per_k * kilo + p.per_round) + p.per_work * kilo * work;
    };
    return static_cast<double>(m / 32) * pass(32) + (m % 32 ? pass(m % 32) : 0);
}

// mm_f32_tiles: 128 x 128 tiles that each walk all of k, 256 of them side by side.
inline double f32_tiles_us(size_t m, size_t k, size_t n, size_t count) {
    const uint64_t tiles = static_cast<uint64_t>((m + 127) / 128) * ((n + 127) / 128) * count;
    return 3.7 + 1e-3 * static_cast<double>(k) * (12.6 + 62.0 * static_cast<double>((tiles + 255) / 256)) + 2.46 * static_cast<double>(tiles) / 256;
}

// mm_generic, up to 16 rows: its own chain of steps through k, or the elements of B.
inline double f32_plain_us(size_t k, size_t n, size_t count) {
    const double chain = 28e-3 * static_cast<double>(k), work = 2.84e-6 * static_cast<double>(k) * static_cast<double>(n) * static_cast<double>(count);
    return 1.6 + (chain > work ? chain : work);
}

enum class F32Route { rows, tiles, plain };

// rows_ok, tiles_ok: the kernels take these operands.  Up to eight rows the tiles, which do the work of 128, are not
// considered: the passes end first from k = 128 on ([8, 4096] x [50257, 4096]^T 151 us in a pass, 536 on the tiles, 545 on
// the plain kernel), the plain kernel below that.
inline F32Route f32_route(size_t m, size_t k, size_t n, size_t count, bool b_is_nk, bool rows_ok, bool tiles_ok) {
    const double rows = rows_ok ? f32_rows_us(m, k, n, count, b_is_nk) : 1e30;
    if (m <= 8) return rows <= f32_plain_us(k, n, count) ? F32Route::rows : F32Route::plain;
    const double tiles = tiles_ok ? f32_tiles_us(m, k, n, count) : 1e30;
    if (!rows_ok && !tiles_ok) return F32Route::plain;
    return rows <= tiles ? F32Route::rows : F32Route::tiles;
}

}  // namespace rg
