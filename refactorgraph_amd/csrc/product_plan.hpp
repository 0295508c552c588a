// What the kernels of MatMul and MatMulInteger are expected to take, and the choice between them: plain functions of
// sizes (no device, no HIP), so that the choice itself is tested on the CPU.  All times are microseconds; the figures are
// least squares over launches of every kernel that takes a call, at sizes drawn over the ranges named with them.
#pragma once

#include <cstddef>
#include <cstdint>
#include <utility>

namespace rg {

// ---------------------------------------------------------------- tiles, one workgroup on a CU
//
// `fixed` us a round of 256 workgroups, and per step of k `alone` ns while few CUs have a tile, `full` ns while all have one
// (they then share what the memory side of the CUs delivers); a launch takes kLaunchUs besides.
struct TileShape {
    uint32_t rows, cols;
    double fixed, alone, full;
};
constexpr uint32_t kPlanCus = 256;

inline uint64_t tile_count(const TileShape &t, size_t m, size_t n, size_t count) {
    return static_cast<uint64_t>((m + t.rows - 1) / t.rows) * ((n + t.cols - 1) / t.cols) * count;
}
inline double tiles_us(const TileShape &t, uint64_t tiles, double steps, double extra_fixed = 0) {
    const double rounds = static_cast<double>(tiles / kPlanCus), left = static_cast<double>(tiles % kPlanCus) / kPlanCus;
    const double fixed = t.fixed + extra_fixed;
    return rounds * (fixed + 1e-3 * steps * t.full) + (left > 0 ? fixed + 1e-3 * steps * (t.alone + (t.full - t.alone) * left) : 0);
}

// ---------------------------------------------------------------- FP16 / BF16
//
// Fitted over 5,900 products of 1 to 2048 rows, k 64 to 11008, 64 to 32000 columns, 1 to 256 of them side by side, both
// layouts of B, with and without a bias.

// mm_ring, steps of 64 k.
constexpr TileShape kRingShapes[] = {{64, 64, 2.7, 145, 300},   {64, 128, 3.4, 210, 440},  {128, 128, 4.2, 360, 580},
                                     {128, 192, 6, 370, 800}, {128, 256, 7.2, 580, 888}, {256, 256, 12.2, 920, 1525}};
constexpr int kRingShapeCount = 6;
constexpr double kRingLaunchUs = 1.0;
// the 256 x 256 tiles store element by element where rows of the output are no whole 16-byte words; the smaller tiles hide that.
// Over 451 products with such rows the plan takes 0.3 % longer than the fastest shape (0.9 with nothing here, 1.8 with 4.7 us:
// 256 products [256, 512] x [1001, 512]^T 149 us on these tiles, 175 on 128 x 256; 16 of [512, 64] x [4099, 64]^T 45 and 42)
constexpr double kRoughStoresUs = 1.5;

struct RingPlan {
    int first, rest;   // shape of the first `columns` columns and of those behind them
    uint32_t columns;  // 0: all on `rest`
    double us;
};

// One shape for the whole product, or whole rounds of one shape and another one for the columns that are left: 344 tiles of
// 256 x 256 ([2048, 4096] x [4096, 11008]) would be a full round and one with two thirds of the CUs idle (208 us); a full
// round over 8192 columns and 240 tiles of 128 x 192 behind it take 171 us.  Over the sizes above the plan takes 0.9 %
// longer than the fastest shape of each product.
inline RingPlan ring_plan(size_t m, size_t k, size_t n, size_t count, bool rough_stores) {
    RingPlan best{0, 0, 0, 1e30};
    const double steps = static_cast<double>(k / 64);
    auto rough = [&](const TileShape &t) { return rough_stores && t.rows == 256 ? kRoughStoresUs : 0.0; };
    auto single = [&](size_t columns) {
        std::pair<int, double> one{0, 1e30};
        for (int i = 0; i < kRingShapeCount; ++i) {
            const TileShape &t = kRingShapes[i];
            const double us = tiles_us(t, tile_count(t, m, columns, count), steps, rough(t));
            if (us < one.second) one = {i, us};
        }
        return one;
    };
    const auto whole = single(n);
    best.rest = whole.first;
    best.us = kRingLaunchUs + whole.second;
    if (count != 1) return best;
    for (int i = 0; i < kRingShapeCount; ++i) {
        const TileShape &t = kRingShapes[i];
        const size_t row_tiles = (m + t.rows - 1) / t.rows, tiles = row_tiles * (n / t.cols);
        const size_t wide = tiles / kPlanCus * kPlanCus / row_tiles;  // columns of tiles in whole rounds
        if (wide == 0 || wide * t.cols >= n) continue;
        const auto rest = single(n - wide * t.cols);
        const double us = kRingLaunchUs + tiles_us(t, row_tiles * wide, steps, rough(t)) + rest.second;
        if (us < 0.97 * best.us) best = {i, rest.first, static_cast<uint32_t>(wide * t.cols), us};
    }
    return best;
}

// Up to 32 rows on the kernels that read the weights once, columns of all products side by side: mm_skinny (B as [n, k]) and
// a pass of mm_rows_kn (B as [k, n]).  With the weights in the caches, as the fit has them, the choice between these and the
// tiles takes 0.3 % longer than the faster one on average, and beyond 32 rows neither ended before the tiles at any size.
// With weights from memory the tiles, which wait for each step's copies, take up to 1.6 times as long and the few-rows kernels
// about what they took: there the rule takes 0.2 % (mm_skinny), 1 % (up to 8 rows of mm_rows_kn) and 3.6 % (9 to 16 rows, whose
// cost is 0.3 us per 1000 of k below the fit for this) longer.  33 to 64 rows stay on the tiles: two slabs of mm_skinny took
// 40 us against 53 from memory and 39 against 32 from the caches ([64, 11008] x [1024, 11008]^T), 20 and 22, 19 and 14.5 at
// [64, 4096] x [4096, 4096]^T; over k from 3072 and 512 to 6144 columns they take 7 % longer than the faster kernel from
// memory and 31 % from the caches, the tiles 10 % and nothing.
inline double skinny_us(size_t k, size_t columns) {
    const double kilo = 1e-3 * static_cast<double>(k), wide = 1e-3 * static_cast<double>(columns);
    return 1.5 + 0.74 * kilo + 0.3 * kilo * wide + 0.21 * wide;
}
inline double rows_kn_us(size_t m, size_t k, size_t n, size_t count) {
    const double kilo = 1e-3 * static_cast<double>(k), wide = 1e-3 * static_cast<double>(n * count);
    // (one product: beyond a workgroup per CU a second round walks k again, [8, 2048] x [2048, 6144] 16.6 us, 13.5 on mm_ring)
    const size_t strips = n % 32 == 0 && n >= 8192 ? n / 32 : (n + 15) / 16;
    const double again = count == 1 ? 0.6 * kilo * static_cast<double>((strips - 1) / kPlanCus) : 0;
    if (m <= 8) return 0.9 + 1.64 * kilo + 0.32 * kilo * wide + 0.28 * wide + again;
    return 2.9 + 1.33 * kilo + 0.334 * kilo * wide + 0.15 * wide + again;  // (9 to 16 rows)
}
// A pass of four rows of mm_gemv_kn: a workgroup's chain through k, or B at what 16-byte pieces of its rows come in at.
inline double gemv_kn_us(size_t m, size_t k, size_t columns) {
    const double chain = 2.5 + 3.1e-3 * static_cast<double>(k), bytes = 2.0 * static_cast<double>(k) * static_cast<double>(columns) / 1.25e6;
    return static_cast<double>((m + 3) / 4) * (chain > bytes ? chain : bytes);
}
// mm_generic, up to 16 rows.
inline double plain_us(size_t k, size_t columns) {
    const double chain = 31e-3 * static_cast<double>(k), work = 2.6e-6 * static_cast<double>(k) * static_cast<double>(columns);
    return 1.5 + (chain > work ? chain : work);
}
// mm_tiles16, steps of 64 k.
inline double tiles16_us(size_t k) { return 4.0 + 0.83 * static_cast<double>((k + 63) / 64); }

enum class HalfRoute { tiles, rows, rows_kn, gemv, gemv_kn, skinny, plain };

// Which kernels take the operands (alignment, layouts, divisibility), with the row counts each is made for.
struct HalfKernels {
    bool ring, tiles16;        // mm_ring; mm_tiles16, which takes what mm_ring takes and more
    bool gemv, rows, skinny;   // B as [n, k]: up to 4, 2 to 16, up to 32 rows
    bool gemv_kn, rows_kn;     // B as [k, n]: up to 32 rows each
};

// `count` products side by side.  One to 16 rows that mm_gemv and mm_rows take read W as [n, k] once: never a tile.
inline HalfRoute half_route(size_t m, size_t k, size_t n, size_t count, bool b_is_nk, const HalfKernels &can, bool rough_stores) {
    const bool tiles = can.ring || can.tiles16;
    if (tiles && m > 32) return HalfRoute::tiles;
    const size_t columns = n * count;
    auto ring_us = [&] { return ring_plan(m, k, n, count, rough_stores).us; };
    if (b_is_nk) {
        if (can.rows) return HalfRoute::rows;
        if (can.gemv) return HalfRoute::gemv;
        if (can.skinny) return can.ring && ring_us() < skinny_us(k, columns) ? HalfRoute::tiles : HalfRoute::skinny;
    } else {
        // 17 rows and more: the tiles, unless the columns are whole groups of 32 workgroups (an XCD then has whole 128-byte
        // pieces of B's k-rows) and few, and B fits the L2s: over 75 such calls the tiles take 1.14 times as long from memory
        // and 1.10 times from the caches ([17, 11008] x [11008, 1024] 52 and 42 us, 31 and 24).  Elsewhere the passes win up to
        // 20 % from memory and lose more from the caches ([24, 4096] x [4096, 768] level, 1.45 times the tiles' time).
        if (can.rows_kn && m > 16) {
            const bool few = count == 1 && n % 512 == 0 && n <= 2048 && static_cast<uint64_t>(k) * n <= 12u << 20;
            return can.ring && !few ? HalfRoute::tiles : HalfRoute::rows_kn;
        }
        if (can.rows_kn) return can.ring && ring_us() < rows_kn_us(m, k, n, count) ? HalfRoute::tiles : HalfRoute::rows_kn;
        if (can.gemv_kn) {
            // (a second pass of four rows never ended before the tiles: [5, 4096] x [4096, 1000] 34 us, 14 on mm_ring)
            if (m <= 4) return HalfRoute::gemv_kn;
            if (can.ring) return HalfRoute::tiles;
            const uint64_t tiles128 = static_cast<uint64_t>((n + 127) / 128) * count;  // (mm_tiles16, one launch of few tiles)
            return can.tiles16 && tiles128 <= 384 && tiles16_us(k) < gemv_kn_us(m, k, columns) ? HalfRoute::tiles : HalfRoute::gemv_kn;
        }
    }
    if (!tiles) return HalfRoute::plain;
    if (m > 8) return HalfRoute::tiles;
    // up to eight rows that no few-rows kernel takes ([8, 3648] x [2376, 3648]^T 123 us on the plain kernel, 14 on mm_ring;
    // 256 products [8, 512] x [1000, 512]^T 303 and 55)
    if (can.ring) return ring_us() < plain_us(k, columns) ? HalfRoute::tiles : HalfRoute::plain;
    return static_cast<uint64_t>(n) * k > 1400000u + 4500u * static_cast<uint64_t>(k) ? HalfRoute::tiles : HalfRoute::plain;
}

// ---------------------------------------------------------------- uint8 / int8
//
// Fitted over 3,600 products of 5 to 4096 rows, k 128 to 11008, 16 to 11008 columns, 1 to 128 of them side by side, every
// form of zero points, int32 and dequantised outputs; over them the choice takes 0.9 % longer than the fastest kernel.

// mmi_ring, steps of 128 k, and mmi_mfma_256x256.
constexpr TileShape kIntegerShapes[] = {{64, 64, 3.2, 245, 330}, {64, 128, 4.5, 350, 660}, {128, 128, 4.8, 580, 770}, {128, 256, 7.7, 570, 1020}};
constexpr int kIntegerShapeCount = 4;
constexpr TileShape kIntegerLargeShape = {256, 256, 7.2, 1250, 1790};
constexpr double kIntegerScaleUs = 1.0;  // a round of mmi_ring with dequantised outputs takes longer by this

// mmi_skinny: tiles of 128 k that a workgroup of 256 columns sums itself, as few as keep about kSkinnyWorkgroups workgroups
// per launch (one per CU; 512 and 128 were measured: slower), and the shares of k that makes.
constexpr uint64_t kSkinnyWorkgroups = 256;
struct SkinnyShares {
    uint32_t tiles, shares;
};
inline SkinnyShares integer_skinny_shares(size_t k, size_t n, size_t count) {
    const uint32_t k_tiles = static_cast<uint32_t>(k / 128);
    uint32_t tiles = static_cast<uint32_t>((static_cast<uint64_t>(k_tiles) * (n / 256) * count + kSkinnyWorkgroups - 1) / kSkinnyWorkgroups);
    tiles = tiles < 1 ? 1 : tiles > k_tiles ? k_tiles : tiles;
    return {tiles, (k_tiles + tiles - 1) / tiles};
}

// mmi_zero, mmi_skinny and, for dequantised outputs, mmi_dequantize_in_place: a workgroup's tiles, one atomic per output and
// share.  More than 128 rows are two passes over B and never ended first.
inline double integer_skinny_us(size_t m, size_t k, size_t n, size_t count, bool dequantize) {
    if (m > 128) return 1e30;
    const SkinnyShares s = integer_skinny_shares(k, n, count);
    const double rounds = static_cast<double>((n / 256) * s.shares * count) / static_cast<double>(kSkinnyWorkgroups);
    const double outputs = 1e-6 * static_cast<double>(m) * static_cast<double>(n) * static_cast<double>(count);
    const double fixed = m <= 32 ? 4.0 : m <= 64 ? 4.5 : 5.5, tile = m <= 32 ? 1.44 : m <= 64 ? 1.98 : 3.23;
    return fixed + (rounds > 1 ? rounds : 1) * tile * s.tiles + 2.0 * outputs * s.shares + (dequantize ? 2.5 + 1.3 * outputs : 0);
}

// What a step of mmi_ring takes longer with weights from memory instead of the caches is 0.1 to 0.24 us; mmi_skinny takes the
// same.  The fits have the caches, so one product's tiles are charged a part of that which serves both kinds of call, where B
// is large (a small one stays in the caches) and mmi_skinny's workgroups have few columns (11008: level from memory, 1.3 times
// the tiles' time from the caches).  Over 1,820 products of 5 to 128 rows the choice takes 1.5 % longer than the faster kernel
// from memory and 1.1 % from the caches (nothing charged: 2.3 and 0.9 %, twice the time at worst; [33, 11008] x [11008, 6144]
// 51 us on the tiles, 26 on mmi_skinny).
inline double integer_from_memory_us(size_t m, size_t k, size_t n, double steps) {
    return static_cast<uint64_t>(k) * n >= 8u << 20 && n <= 6144 ? steps * (m <= 32 ? 0.02 : 0.07) : 0;
}

struct IntegerRoute {
    enum { ring, large, skinny } kernel;
    int shape;  // of mmi_ring
};

// For operands that mmi_ring takes; large_ok, skinny_ok: the other two take them as well.
inline IntegerRoute integer_route(size_t m, size_t k, size_t n, size_t count, bool dequantize, bool large_ok, bool skinny_ok) {
    const double steps = static_cast<double>((k + 127) / 128);
    IntegerRoute best{IntegerRoute::ring, 0};
    double us = 1e30;
    for (int i = 0; i < kIntegerShapeCount; ++i) {
        const double t = 0.4 + tiles_us(kIntegerShapes[i], tile_count(kIntegerShapes[i], m, n, count), steps, dequantize ? kIntegerScaleUs : 0);
        if (t < us) us = t, best = {IntegerRoute::ring, i};
    }
    if (large_ok && 0.4 + tiles_us(kIntegerLargeShape, tile_count(kIntegerLargeShape, m, n, count), steps) < us) return {IntegerRoute::large, 0};
    if (count == 1) us += integer_from_memory_us(m, k, n, steps);
    if (skinny_ok && integer_skinny_us(m, k, n, count, dequantize) < us) return {IntegerRoute::skinny, 0};
    return best;
}

// ---------------------------------------------------------------- F32
//
// Fitted over 2,500 products of 1 to 256 rows, k 64 to 8320, 16 to 50257 columns: the cheaper one by these costs takes 0.06 %
// longer than the faster kernel of each call.

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

enum class F32Route { rows, tiles, plain };

// rows_ok, tiles_ok: the kernels take these operands.  Up to eight rows the tiles, which do the work of 128, are not
// launched and so not weighed either ([8, 4096] x [50257, 4096]^T 151 us in a pass, 545 on the plain kernel).  Beyond, the passes
// where they are expected to end first, and where they lose little: their sums are 16 partial sums of k each, a tile's are one
// chain (0.9e-7 and 4e-7 from 64 bits at k = 512), so the tiles have to win on costs that flatter the passes too (27 us for 32 rows
// against 4096 x 4096, 300 us for up to 768 tiles at k = 4096).
inline F32Route f32_route(size_t m, size_t k, size_t n, size_t count, bool b_is_nk, bool rows_ok, bool tiles_ok) {
    if (m <= 8) return rows_ok ? F32Route::rows : F32Route::plain;
    if (!rows_ok) return tiles_ok ? F32Route::tiles : F32Route::plain;
    if (!tiles_ok || f32_rows_us(m, k, n, count, b_is_nk) <= f32_tiles_us(m, k, n, count)) return F32Route::rows;
    const double weights = static_cast<double>(n) / 4096 * static_cast<double>(k) / 4096;
    const double tiles = static_cast<double>(((m + 127) / 128) * ((n + 127) / 128));
    const double passes = static_cast<double>((m + 31) / 32) * (3.0 + (b_is_nk ? 27.0 : 33.0) * weights);
    return passes <= 3.0 + 300.0 * static_cast<double>(k) / 4096 * static_cast<double>((static_cast<uint64_t>(tiles) + 767) / 768) ? F32Route::rows : F32Route::tiles;
}

}  // namespace rg
