// Which linears and batches run on the row tiles (qxt_q4_0_rows.hip), and the
// launch plan of a batch: waves of a workgroup, LDS, and column tiles per
// workgroup by the length of K.  Host code only, without HIP.
#pragma once

#include <algorithm>
#include <cstddef>
#include <map>

namespace qxt {

constexpr int kRowsWaves = 8;            // most waves of a workgroup
constexpr int kRowsWavesPerCu = 12;      // resident by registers
constexpr int kRowsMaxPasses = 4;        // chunks per wave and tile
constexpr size_t kRowsLds = 160 * 1024;
constexpr size_t kRowsChunkBytes = 6656;  // staged activation of a chunk (32 blocks of four rows)
constexpr size_t kRowsSumBytes = 256;     // running sums of a tile

struct RowsPlan {
    int waves;    // of a workgroup
    size_t lds;
    bool groups;  // workgroups compute waves / chunks column tiles side by side where K has fewer chunks
    int steps;    // column tiles one after the other
    bool evened;  // fewer of them for a K of more passes
    int fewest_passes;

    int groups_of(int chunks) const { return groups ? std::max(1, waves / chunks) : 1; }
    int passes_of(int chunks) const { return (chunks + waves - 1) / waves; }
    // Columns of a workgroup over a K of so many chunks.
    int columns(int chunks) const {
        return 16 * groups_of(chunks) * (evened ? std::max(1, steps * fewest_passes / passes_of(chunks)) : steps);
    }
};

// Column tiles (16 columns) of a batch by the chunks of their K.
using RowsTiles = std::map<int, long>;

// Waves for `chunks` chunks of K alone: as few passes as fit.
inline int rows_waves(int chunks, int most_waves) {
    const int passes = (chunks + most_waves - 1) / most_waves;
    return (chunks + passes - 1) / passes;
}

// Workgroups a CU holds at once.
inline long rows_resident(int waves, int waves_per_cu, size_t lds) {
    return std::max<long>(1, std::min<long>(waves_per_cu / waves, static_cast<long>(kRowsLds / lds)));
}

// Column tiles that a workgroup takes one after the other (they share a staged
// activation), for a grid of `steps` such steps over `slots` resident
// workgroups: one while the chip holds every workgroup at once, two where that
// makes one round of them, and for larger grids up to three as long as several
// rounds remain to even out the last.
inline int rows_steps(long steps, long slots) {
    if (steps <= slots) return 1;
    if (steps <= 2 * slots) return 2;
    return static_cast<int>(std::min<long>(3, std::max<long>(1, steps / (4 * slots))));
}

// Whether a batch takes the row tiles; the v_dot4 batch kernel has the rest
// (MI355X, two rows, us there / here).  Units: 8 blocks of one column.
//   * A K below 1024 leaves most of a chunk empty, which many tiles pay for: eight
//     linears of 32000 columns over K = 256 and eight of 2048 over K = 2048 18.8 /
//     28.0; of 4096 over 256 and 2048 over 512, fp32 rows, 7.7 / 10.0 (both use
//     a third of their chunks), but one of each 6.3 / 5.1.
//   * The passes over a very long K follow one another in a small grid: 4096
//     columns of K = 1024 beside 128 of K = 24576 15.7 / 17.9.  Given as fp32 rows,
//     which are quantised in less time here, 55.6 / 22.6.
inline bool rows_batch_preferred(const RowsTiles &tiles, double units, bool fp32_rows, int cus) {
    double chunks = 0.0;
    long total = 0;
    for (const auto &[c, n] : tiles) chunks += static_cast<double>(n) * c, total += n;
    const int most = tiles.rbegin()->first;
    if (units < 0.4 * 64 * chunks && most <= kRowsWaves && total > 8L * cus) return false;
    return fp32_rows || most < 20 || chunks >= 4.0 * cus;
}

inline RowsPlan rows_batch_plan(const RowsTiles &tiles, int cus) {
    constexpr int kBusy = 9;  // waves that keep a CU issuing
    const int most = tiles.rbegin()->first;
    int least = 1 << 30;
    for (const auto &[chunks, n] : tiles) least = std::min(least, rows_waves(chunks, kRowsWaves));
    auto bytes_of = [&](int waves, bool grouped) {
        size_t bytes = 0;
        for (const auto &[chunks, n] : tiles)
            bytes = std::max(bytes, chunks * kRowsChunkBytes +
                                        static_cast<size_t>(grouped ? std::max(1, waves / chunks) : 1) * kRowsSumBytes);
        return bytes;
    };
    auto slots_of = [&](int waves, bool grouped) {
        return cus * rows_resident(waves, kRowsWavesPerCu, bytes_of(waves, grouped));
    };
    // Time of a plan in steps of one chunk on a busy CU: the passes of the
    // longest K, or the chunks of the whole grid over the waves that have one if
    // that is more, with a twentieth for each further pass (the last may be short)
    // and a tenth for a CU with a single workgroup, whose waves all wait for the
    // same turns.
    auto cost_of = [&](int waves, bool grouped) {
        const long slots = slots_of(waves, grouped);
        double sum = 0.0;
        for (const auto &[chunks, n] : tiles) {
            const int passes = (chunks + waves - 1) / waves;
            const double working = passes > 1 ? static_cast<double>(chunks) / passes
                                   : grouped  ? waves / chunks * chunks
                                              : chunks;
            sum += static_cast<double>(n) * chunks * (0.95 + 0.05 * passes) /
                   std::min(static_cast<double>(kBusy) * cus, slots * working);
        }
        return std::max(0.6 * ((most + waves - 1) / waves), sum) * (1.0 + 0.1 * cus / slots);
    };
    // The waves that the shortest K needs (a longer one takes more passes):
    // waves without a chunk would idle.  K = 2048 and 5632 together, the
    // 154-linear step at two rows: six waves 222 us, two 139.
    const int fewest = (most + kRowsMaxPasses - 1) / kRowsMaxPasses;
    RowsPlan plan{};
    plan.waves = std::max(least, fewest);
    // Not where K differs so that they leave the chip waiting.  One LDS size
    // serves the whole launch, so a long K leaves few workgroups to a CU: these
    // then need more waves than a short K has chunks, and groups to use them all.
    // Whole layers of hidden / feed-forward K on MI355X, two fp32 rows, lane
    // weights, us with the shortest K's waves and task order, and so: twenty of
    // 512 / 16384 421 -> 112, of 512 / 8192 102 -> 46, of 1024 / 8192 126 -> 69,
    // of 2048 / 5632 130 -> 121; six of 2048 / 16384 215 -> 113 (v_dot4 batch
    // kernel: 205, 69, 131, 166, 247).
    double best = cost_of(plan.waves, false) / 1.1;
    for (int w = fewest; w <= kRowsWaves; ++w)
        for (const bool grouped : {false, true})
            if (cost_of(w, grouped) < best) best = cost_of(w, grouped), plan.waves = w, plan.groups = grouped;
    const long slots = slots_of(plan.waves, plan.groups);
    long all = 0;
    for (const auto &[chunks, n] : tiles) all += n;
    plan.groups = plan.groups && all > slots;
    plan.lds = bytes_of(plan.waves, plan.groups);
    plan.fewest_passes = plan.passes_of(tiles.begin()->first);
    auto workgroups = [&] {
        long sum = 0;
        for (const auto &[chunks, n] : tiles) sum += (16 * n + plan.columns(chunks) - 1) / plan.columns(chunks);
        return sum;
    };
    // As many steps for every K, but fewer for one of more passes where the chip
    // holds every workgroup then too.
    plan.steps = 1;
    plan.steps = rows_steps(workgroups(), slots);
    plan.evened = true;
    plan.evened = workgroups() <= slots;
    return plan;
}

// Which single linears of 2 to 15 rows take the row tiles, by what was measured
// faster on MI355X (us, the other kernels -> these; back to back over rotated
// weights).  Fitted to 8,100 shapes (25 K from 256 to 16384 x 18 N from 64 to
// 32000 x 9 row counts x both layouts): 1.36 times the others in the geometric
// mean, ten shapes more than 4 % slower, by at most 1.07, where taking every shape
// leaves 1,588; on 3,360 others 1.34 times, 13 slower, by at most 1.35 (4 rows,
// lanes, 6400 x 9216).  K x N below; `n` is column tiles per 256 CUs.  The other
// kernels: q4_0_mfma4 (four-row tiles, K <= 4096 with 16 % (K / 256) == 0),
// q4_0_stream (native rows, blocks over lanes), v_dot4 tiles.
//   * Many tiles: the others stream the weights with more of them in flight,
//     these are bound by instructions (lanes, 2 rows, 4608 x 32000 21.3 -> 45.2;
//     but from K = 14336 their staged rows leave them one workgroup a CU:
//     16384 x 8192 39.2 -> 26.3).
//   * Just over one tile per CU these take a second round (lanes, 3 rows,
//     4608 x 4608 8.4 -> 12.0; native, 4 rows, 14336 x 4608 15.7 -> 23.4).
//   * Few tiles over a long K: the others spread it over the chip, these keep it
//     to a workgroup per 16 columns (native, 5 rows, 8192 x 1024 6.9 -> 9.1,
//     6144 x 64 3.9 -> 6.9; lanes 14336 x 64 9.0 -> 11.1).
inline bool rows_linear_takes(bool lanes, int rows, int blocks, long tiles, long cus) {
    const int b = blocks;
    const long n = tiles * 256 / cus;
    const bool mfma4 = b <= 128 && 16 % (b / 8) == 0;
    const bool just_over = n > 256 && n <= 320;
    const bool three = rows > 8 && rows <= 12;  // three rows a lane, the others' third round of four
    if (b < 16 && n > 512) return three;        // three quarters of each chunk are empty
    if (lanes) {
        if (rows <= 3) {
            // 2048 x 256 4.3 -> 3.3, 2048 x 8192 5.9 -> 5.6; 4096 x 4096 6.4 -> 5.7; 2 rows
            // 5632 x 2048 6.9 -> 6.4, 11008 x 4096 15.8 -> 12.5; 3 rows 8192 x 8192 19.1 -> 15.1.
            if (b <= 64) return n <= 512;
            if (b <= (rows == 2 ? 176 : 224)) return n <= 256 || (b > 192 && n > 320 && n <= 512);
            if (rows == 2) return b >= 448 ? n >= 192 : b > 256 && n > 192 && n <= 256;
            return b >= 256 && n >= 256 && !(b <= 352 && just_over);
        }
        if (rows == 4) {
            // 2048 x 256 4.3 -> 3.4, 2304 x 6000 6.9 -> 5.4, 5632 x 2048 7.3 -> 6.4,
            // 5120 x 16384 28.5 -> 20.7, 8192 x 4096 10.8 -> 9.5.
            if (mfma4) return n <= (b <= 64 ? 128 : 32);
            if (b <= 128) return true;
            if (b <= 192) return n <= 256 || (b >= 160 && n > (b == 192 ? 640 : 768) && n <= 1280);
            return (b <= 224 || n >= 128) && !(b <= 352 && just_over);
        }
        // 8 rows: 4096 x 4096 7.0 -> 6.4, x 11008 18.2 -> 12.2, 2048 x 5632 6.1 -> 5.9,
        // 2048 x 16384 8.8 -> 9.8 (not taken), 11008 x 4096 32.1 -> 14.6.
        if (b >= 256 && n <= (rows <= 8 ? 32 : three ? 14 : 16)) return false;
        if (rows <= 8 && b == 64) return n <= 512 || n > 1024;
        if (rows <= 8 && b == 128) return n <= 256 || n > 512;
        return !(rows <= 8 && b > 128 && b <= 192 && just_over);
    }
    if (rows <= 4) {
        // 2048 x 256 4.2 -> 3.2, x 5632 5.6 -> 4.8; 4 rows 11008 x 4096 13.4 -> 11.4,
        // but x 4608 14.7 -> 18.0 (not taken).
        if (b <= 64) return n <= 512;
        if (rows < 4) return false;
        if (b <= 128) return !mfma4 && n <= 512;
        return b > 256 && b < 416 && n >= 256 && !(n > 256 && n <= 358);
    }
    // 8 rows: 2048 x 5632 6.2 -> 5.6, 4096 x 4096 7.5 -> 6.1, x 11008 16.0 -> 12.7,
    // 11008 x 4096 22.3 -> 13.0; 9 rows 14336 x 4608 35.3 -> 42.4 (not taken).
    if (b <= 64) return true;
    if (b > 496 && !(rows > 12 && n <= 256)) return false;
    if (b >= 416 && three && n > 256 && n < 1024) return false;
    if (just_over && (b <= 128 || (rows <= 8 && b >= 192 && b <= 216) || (three && b >= 336))) return false;
    // Least tiles, by K, up to eight rows and past them.
    const bool few = rows <= 8;
    if (b <= 112) return n >= (few ? 32 : 16);
    if (b <= 176) return n >= (few ? 96 : 64);
    if (b <= 224) return n >= (few ? 128 : 96);
    if (b <= 256) return n >= (few ? 256 : 128);
    if (b < 416) return n >= (few ? 128 : 64);
    return n >= (few ? 192 : 96);
}

// Sixteen or more rows over lane weights, which the prefill tiles do not read:
// the other kernels take four rows at a time and read the weights again for each
// four, these sixteen or eight.  MI355X, us, those -> these: 24 rows 2048 x 32000
// 52 -> 32, 96 rows 4096 x 4096 53 -> 25, 512 rows 2048 x 5632 181 -> 59; but 16 rows
// 14336 x 64 9.3 -> 11.2, 64 rows 256 x 11008 7.6 -> 9.9 (few tiles of a long K, many
// of a K that fills a quarter of a chunk: not taken).
inline bool rows_lanes_prefill_takes(int rows, int blocks, long tiles, long cus) {
    const long n = tiles * 256 / cus * ((rows + 15) / 16);
    return blocks < 16 ? n <= 640 : blocks < 256 || n > 8;
}

}  // namespace qxt
