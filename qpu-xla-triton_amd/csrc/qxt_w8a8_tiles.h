// Tiles of the int8 GEMM below 256 x 256 ones (qxt_w8a8.hip).  Host code only,
// without HIP.
#pragma once

namespace qxt {

// w8a8_gemm_kernel instantiations.  Groups: K split over groups of waves inside
// the workgroup; Short: K stages of 64 bytes, three workgroups to a CU.
enum class MidTile {
    k128x128Short,
    k128x128,
    k128x128Groups,
    k128x64Groups,
    k32x32Groups,
    k64x32Groups,
    k64x64Groups,
    k64x64,
};

// Tiles of problems too small for 256 x 256 ones.  What bounds them is what a CU
// takes in from L2, measured at 55 to 61 bytes per ns with any of these tiles,
// so the choice is the largest tile that still gives (nearly) every CU one, with
// at least two K stages in flight in registers: one stage in flight left each
// stage waiting for L2 (0.6 us at 64 x 64).  Two groups of four waves per tile
// (KS = 2) where a CU holds one workgroup.
// Measured on MI355X, GEMM alone, rotated weights, back to back (M x K x N, us;
// before: 128 x 128 tiles from one tile per CU, else 64 x 64, one stage in
// flight):
//   128 x 128:  512 x 4096 x 14336 55.8 -> 46.5, 1024 x 4096 x 8192 53.2 -> 48.9;
//               KS = 2: 1024 x 4096 x 4096 44.7 -> 26.9, 256 x 4096 x 14336 36.4 -> 27.2,
//               256 x 4096 x 11008 (172 tiles) 32.9 -> 26.2; at 141 tiles 23.7
//               against 21.7 with 64 x 64;
//   128 x 64:   512 x 14336 x 4096 89.5 -> 51.7 (64 x 64: 62.3), 512 x 4096 x 4096
//               27.2 -> 18.4; a second round of them (282 tiles) 28.3 against 21.7;
//   64 x 64:    KS = 2, three stages: 48 x 4096 x 14336 29.1 -> 14.8, 128 x 14336 x
//               4096 87.4 -> 34.4, 8 x 14336 x 4096 89.0 -> 27.4, 32 x 4096 x 11008
//               28.3 -> 11.8; past one tile per CU, KS = 1: 300 x 4096 x 6000
//               29.6 -> 21.7, 64 x 1024 x 32000 13.1 -> 9.7, 768 x 2048 x 5632
//               24.1 -> 20.2 (128 x 128: 24.4).
// While even 32 x 32 tiles, or 64 x 32, leave at most one to a CU they take the
// call from K = 1024: a CU takes in half of the columns or less, and eight or
// four groups of waves (KS) keep as many loads in flight.  64 x 64 -> 32 x 32:
// 8 x 14336 x 4096 27.9 -> 21.0, 48 x 14336 x 4096 33.4 -> 22.5, 16 x 14336 x 512
// 26.7 -> 16.1, 8 x 4096 x 4096 10.4 -> 8.6, packed 8 x 14336 x 4096 48.0 -> 22.2; 512 of
// K 3.8 -> 4.6, a second round of tiles (8 x 4096 x 8800) 13.0 -> 16.7, not taken.
// 64 x 64 -> 64 x 32: 128 x 14336 x 4096 35.4 -> 27.8, 200 x 4096 x 2048 10.5 -> 8.9,
// 40 x 8192 x 8192 24.1 -> 19.2; a second round (64 x 4096 x 11008) 16.4 -> 20.7.
// packed: [K / 4, N] weights.
inline MidTile w8a8_mid_tile(long m, long n, long k, bool packed, long cus) {
    auto tiles = [&](long bm, long bn) { return ((m + bm - 1) / bm) * ((n + bn - 1) / bn); };
    const long t128 = tiles(128, 128), t12864 = tiles(128, 64), t64 = tiles(64, 64);
    if (m > 64) {  // fewer rows would leave half of a 128-row tile empty
        // Stages of 64 instead of 128 bytes: over packed weights of a short K,
        // whose transposing LDS writes make the longer stage dearer (2048 x 2048 x
        // 5632 68.1 against 69.8 us), and where three workgroups of them to a CU
        // make one round of what two do not (1536 x 512 x 5632 20.3 -> 16.3,
        // 1536 x 2048 x 5632 38.8 -> 33.9).
        const bool one_round = t128 > 2 * cus && t128 <= 3 * cus && k < 8192;
        if (t128 > cus && !(k < 3072 && 4 * t128 <= 5 * cus))
            return (packed ? k < 3072 : one_round) ? MidTile::k128x128Short : MidTile::k128x128;
        // Two groups of 128 x 128 have to pay for a half-empty chip and their
        // first stages: not over a short K (512 x 512 x 5632 8.6 -> 7.0 with 64 x 64,
        // packed 65 x 512 x 32000 13.5 -> 11.9), nor with packed weights, whose
        // transposing writes take the time twice, while 64 x 64 ones make one round
        // (768 x 4096 x 4096 47.2 -> 38.7; past it 200 x 14336 x 14336 147 against 161).
        if (t128 <= cus && (packed ? k >= 3072 && t64 > 3 * cus
                                   : k >= 1536 && 8 * t128 >= (k < 2048 ? 7 : 5) * cus))
            return MidTile::k128x128Groups;
        // (512 of K, rows 128 to 1024: up to 1.15 times 64 x 64.)
        if (k >= (packed ? 512 : 1024) && t12864 <= cus && 5 * t12864 >= 4 * cus)
            return MidTile::k128x64Groups;
    }
    if (k >= 1024 && tiles(32, 32) <= cus) return MidTile::k32x32Groups;
    if (k >= 1024 && tiles(64, 32) <= cus) return MidTile::k64x32Groups;
    // (256 of K is two stages: 1.1 times one group of waves.)
    if (t64 <= cus && k >= 512) return MidTile::k64x64Groups;
    return MidTile::k64x64;
}

}  // namespace qxt
