// Launch plan of a batch on the row tiles (qxt_q4_0_rows.hip): waves of a
// workgroup, LDS, and column tiles per workgroup by the length of K.  Host
// code only, without HIP.
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

}  // namespace qxt
