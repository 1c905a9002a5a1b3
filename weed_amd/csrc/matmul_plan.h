// Which tile, k ranges and strips a product takes, and which workgroup takes which tile: arithmetic on sizes, shared by the launch
// code and the kernels of matmul.hip and the CPU test of both (tests/plan_check.cpp).
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>

#if defined(__HIPCC__)
#define MM_HD __host__ __device__ __forceinline__
#else
#define MM_HD inline
#endif

namespace weedmm {

constexpr uint32_t kTile = 128; // rows and columns of a tile of the matrix-core kernels
constexpr uint32_t kBig = 256;  // of the larger one of the split-operand kernel
constexpr uint32_t kSlice = 32; // k per slice of the split-operand kernel

inline uint32_t tiles_of(uint32_t n, uint32_t tile) { return (n + tile - 1) / tile; }

// Workgroup -> tile of rows, tile of columns, k range or product of a batch (z).  Workgroups go to the eight XCDs in turns; an XCD
// takes a run of neighbouring tiles, in bands of eight tiles of rows walked column by column, so that those it has in flight
// share operands in its own L2.  Fewer than kPlaced workgroups are a three-dimensional grid in its own order: they all run at once and
// reread little, and the divisions below take part of a microsecond (384 x 768 x 1024 18.4 us on the grid and 20.0 placed, 253 x
// 1728 x 1408 23.2 and 27.4; 512 of them, 1000 x 4096 x 4096 in two ranges: 179.7 and 170.9).
constexpr uint32_t kPlaced = 512;
MM_HD void split_place(uint32_t wg, uint32_t wgs, uint32_t m_tiles, uint32_t n_tiles, uint32_t &mt, uint32_t &nt, uint32_t &z)
{
    const uint32_t xcd = wg & 7, each = wgs / 8, more = wgs % 8;
    const uint32_t at = xcd * each + (xcd < more ? xcd : more) + wg / 8, plane = m_tiles * n_tiles;
    z = at / plane;
    const uint32_t u = at - z * plane, first = u / (8 * n_tiles) * 8, left = m_tiles - first, height = left < 8U ? left : 8U;
    const uint32_t in = u - first * n_tiles;
    nt = in / height;
    mt = first + in - nt * height;
}

// Whole sums of few k are mostly prologue and write-out, which a third workgroup per compute unit overlaps, but it costs registers and
// reads of the LDS: not worth it where two per unit are all that there are (4096 x 64 x 2048, 512 tiles, 13.2 us with two and 13.7
// with three, 2000 x 128 x 2000 13.4 and 13.9), and worth most where the last of them are a round of their own: 3104 x 64 x 2624,
// 525 tiles, 19.7 and 16.0 us, 2200 x 128 x 3900 row-major 29.5 and 24.6, 6000 x 128 x 4000 49.5 and 45.1, 10000 x 100 x 10000 190
// and 165.  (160 k and more have longer slices to wait for, and two of these multiply faster.)
constexpr uint32_t kShortK = 128;
inline bool three_per_unit(uint32_t K, uint32_t k_per_split, uint32_t wgs) { return !k_per_split && K <= kShortK && wgs > 512; }

// Into how many ranges to split k over workgroups (1: not at all) on the fp32 instruction, and of split operands below 2^30
// multiply-adds (plan_tiles has the larger ones).  The tiles run in rounds of two per compute unit,
// each of k / splits slices plus a fixed part per workgroup (prologue, write-out: about 128 slices' worth), and a second
// kernel adds the ranges.  So 128 tiles gain from four ranges (512 x 4096 x 4096: 308 us whole on the fp32
// instruction, 184 in two ranges; with split operands 143 in two and 108 in four), 256 tiles from two (1024 x 4096 x
// 4096: 235 -> 204 us), and 512 tiles from none.
// Ranges of down to 64 k where tiles are few: a workgroup's slices follow each other, each with a trip to memory
// (232 x 768 x 768 51 -> 15 us, 512 x 512 x 512 32 -> 14, 75 x 820 x 691 78 -> 16, 2048 x 768 x 768 47 -> 29; ranges of at
// least 256, which was the rule, left 100 x 1024 x 1024 at 22 us for 14).  Below 448 k the write-out and the sum of many
// tiles' ranges outweigh what they save: 1024 x 1024 x 256 (64 tiles) 18.5 us whole and 20.2 in four ranges, 2048 x 768 x 320
// 22.2 and 24.4, but 768 x 768 x 256 (36 tiles) 18.6 and 16.1.
inline uint32_t choose_k_splits(uint64_t out_tiles, uint32_t K)
{
    if (out_tiles > 512 || (K < 448 && out_tiles > K / 5)) {
        return 1;
    }
    const auto cost = [&](uint32_t s) {
        // (two workgroups share a compute unit and fill each other's barrier waits: together they take 1.5 times
        // what one alone takes -- 1024 x 4096 x 4096, 256 tiles: 235 us whole, 204 in two ranges)
        const double wgs = (double)(out_tiles * s);
        const double rounds = std::ceil(wgs / 512.0), crowd = wgs <= 256.0 ? 1.0 : 1.5;
        return rounds * crowd * ((double)K / s + 128.0) + (s > 1 ? 40.0 + 0.3 * (double)(s * out_tiles) : 0.0);
    };
    uint32_t best = 1;
    double best_cost = cost(1) * 0.92; // (a split has to gain something beyond what two measurements differ by)
    for (uint32_t s = 2; s <= std::min(64U, K / 64U); ++s) {
        if (cost(s) < best_cost) {
            best_cost = cost(s);
            best = s;
        }
    }
    return best;
}

// How a product of split operands of 2^30 multiply-adds and more goes: the tile, and the k ranges (k_per_split 0: whole sums), from
// what its workgroups take in microseconds.  A round of 512 tiles of 128 x 128 (two workgroups per compute unit; up to 256 of them
// take 0.8 of a round) or of 256 tiles of 256 x 256 takes so much per k and something for its start and write-out; partial sums
// are written, read and added at 3.6 GB per millisecond.  The rates are a least-squares fit to 65 products of 65 to 4096 rows in up
// to eleven splits each; `off_grid` is GUARD 2, whose loads and magnitudes cost a little more.  Of 49 products drawn afterwards it is
// within 5 % for 38 and within 10 % for 48 (1994 x 1088 x 896 takes 37 us for 44), and what it chooses is within 3 % of the fastest
// tile and ranges in all but 1051 x 512 x 3136 off the grid (43.4 us whole, 37.4 in two ranges), 3324 x 2496 x 5248 (528, 500 in
// three) and 2221 x 12800 x 1088 (370 in three, 358 in six).
// Beside the rule for 128 x 128 tiles alone that stood here, which counted rounds of 256 and left more than 512 tiles whole: 1649 x
// 5632 x 5824 851 -> 595 us, 556 x 5075 x 13240 788 -> 528, 1906 x 13504 x 9344 3198 -> 2432, 2036 x 1280 x 1984 80 -> 68,
// 2364 x 689 x 1269 58 -> 46, 4096^3 632 -> 572.
constexpr size_t kMostPartials = 256u << 20; // bytes of partial results that a plan may ask for
struct TilePlan {
    uint32_t tile, splits, k_per_split;
    double us;
};
inline TilePlan plan_tiles(uint32_t M, uint32_t N, uint32_t K, uint32_t batch, uint32_t most, bool off_grid)
{
    TilePlan best{ kTile, 1, 0, 0.0 };
    for (uint32_t tile : { kTile, kBig }) {
        // (256 x 256: not for short sums, which are all write-out; 8000 x 128 x 2000, eight products: 238 and 278 us)
        if (tile == kBig && K < 512) {
            break;
        }
        const double tiles = (double)tiles_of(M, tile) * tiles_of(N, tile) * batch;
        const double slots = tile == kBig ? 256.0 : 512.0;
        const double per_k = tile == kBig ? (off_grid ? 0.140 : 0.1365) : (off_grid ? 0.0785 : 0.0712);
        for (uint32_t s = 1; s <= std::max(1U, std::min({ most, 64U, K / (tile / 2) })); ++s) {
            const uint32_t k = s == 1 ? K : ((K + s - 1) / s + kSlice - 1) / kSlice * kSlice;
            if (s > 1 && ((K + k - 1) / k != s || sizeof(float) * (double)s * M * N > (double)kMostPartials)) {
                continue;
            }
            const double wgs = tiles * s, full = std::floor(wgs / slots), rest = wgs - full * slots;
            const double rounds = full + (rest == 0.0 ? 0.0 : (tile != kBig && rest <= 256.0 ? 0.8 : 1.0));
            const double us = 6.0 + rounds * (per_k * k + 2.5) + (s > 1 ? 3.0 + 4.0 * (s + 1) * (double)M * N / 3.6e6 : 0.0);
            if (best.us == 0.0 || us < 0.98 * best.us) { // (more than two runs of one plan differ by)
                best = { tile, s, s == 1 ? 0U : k, us };
            }
        }
    }
    return best;
}

// The rows and columns of a product's whole tiles (see has_strips).
inline uint32_t interior_rows(uint32_t M) { return M / kTile * kTile; }
inline uint32_t interior_cols(uint32_t N)
{
    // (a strip of under 17 columns has no matrix-core kernel: one more tile goes with it; one of under 17 rows is the skinny kernels'
    // own shape)
    return N / kTile * kTile - (N % kTile && N % kTile <= 16 ? kTile : 0U);
}
// Ragged sizes around an interior of whole tiles (a prefill of 1000 tokens): one launch takes the interior, the strips behind it go the
// way their own shapes call for.  Never below 2^32 multiply-adds.
inline bool has_strips(uint32_t M, uint32_t N, uint32_t K, uint32_t batch)
{
    return batch == 1 && M >= kTile && N >= 2 * kTile && (M % kTile || N % kTile) && (uint64_t)M * N * K >= (1ull << 32);
}
// On the fp32 instruction, in rounds of 256 tiles: a strip's few tiles split k and fill the part, plus what its launch costs.
inline bool strips_pay_in_rounds(uint32_t M, uint32_t N)
{
    const uint32_t rows = interior_rows(M), cols = interior_cols(N);
    const auto tiles = [](uint32_t m, uint32_t n) { return (double)tiles_of(m, kTile) * tiles_of(n, kTile); };
    const double whole = std::ceil(tiles(M, N) / 256.0);
    double split = std::ceil(tiles(rows, cols) / 256.0);
    if (rows < M) split += tiles(M - rows, N) / 256.0 + 0.15;
    if (cols < N) split += tiles(rows, N - cols) / 256.0 + 0.15;
    return split < whole;
}
// What they take by plan_tiles: the interior's loads need no guards for addresses off the 16-byte grid.  (Up to 64 rows stream the
// weight, at 3 TB/s and less, where its columns are contiguous along k.)
inline double strips_us(uint32_t M, uint32_t N, uint32_t K, bool b_along_k, uint32_t most, bool off_grid)
{
    const uint32_t rows = interior_rows(M), cols = interior_cols(N);
    const auto part = [&](uint32_t m, uint32_t n) {
        if (!m || !n) {
            return 0.0;
        }
        return m <= 64 && b_along_k && K >= 256 ? 8.0 + 4.0 * (double)K * n / 3.0e6 : plan_tiles(m, n, K, 1, most, off_grid).us;
    };
    return plan_tiles(rows, cols, K, 1, most, false).us + part(M - rows, N) + part(rows, N - cols);
}
// Strips rather than one launch as planned (a tie goes to the one launch).
inline bool strips_beat(const TilePlan &plan, uint32_t M, uint32_t N, uint32_t K, bool b_along_k, uint32_t most, bool off_grid)
{
    return strips_us(M, N, K, b_along_k, most, off_grid) < 0.97 * plan.us;
}

} // namespace weedmm
