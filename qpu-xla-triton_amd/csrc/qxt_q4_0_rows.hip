// Q4_0 x Q8_0 block-dot linear for two or more rows on 16 x 16 matrix-core
// tiles (gfx950): decode batches, short prompts, and batches of linears.
//
// Arithmetic as in qxt_q4_0.hip: per block an exact int32 dot, then
// fl32(fl32(float(dot) * dw) * da), summed in block order.
//
// One wave computes 16 columns x up to 4 RPL rows over a chunk of 32 blocks.
// Lane (kg = lane / 16, n = lane % 16) loads one 144-byte unit (8 blocks) of
// column n, unit kg of the chunk, as nine 16-byte loads; v_permlane16_swap /
// v_permlane32_swap transpose the four nibble words of each block across the
// four lanes of a column, so that lane (kg, n) ends with word kg of every
// block: elements 4 kg .. + 3 (low nibbles) and 16 + 4 kg .. + 3 (high), one
// operand of v_mfma_i32_16x16x32_i8.  A nibble enters as the int8
// 16 (code - 8) -- the nibble in the high half of its byte, its top bit
// flipped -- so no sum of activations is needed; the dot is 16 times the
// block's and dw / 16 (exact: an fp16 value over a power of two) scales it to
// the same fl32(float(dot) * dw).
//
// Activation row r sits in matrix row 4 (r % 4) + r / 4, so output register i
// of lane kg is row kg + 4 i: RPL = ceil(rows / 4) registers of every lane are
// rows in use, and four rows cost one convert, two multiplies and one add per
// block and wave instead of four.
//
// The waves of a workgroup take consecutive chunks of K.  Each keeps its block
// terms in registers; then the waves add them in turn to the tile's running
// sums (LDS), which keeps the block order.  A workgroup walks several column
// tiles where the grid is large, the next tile's weights in flight while a
// tile is computed; its activation rows are staged in LDS once.  In a batch
// whose longest K asks for more waves than a task has chunks, the task's
// workgroups compute waves / chunks column tiles side by side.
//
// What bounds it: small grids, the instructions of one wave (about 450 per
// chunk of 32 blocks at one row per lane, 6 to 7 cycles each with one wave per
// SIMD) and the waves' turns; large grids, those instructions on every SIMD.
// Measured on MI355X against the kernels it replaces (bit-identical): single
// linears at rows_linear_takes (qxt_q4_0_rows_plan.h); a staged decode step of four rows over Llama-7B
// class layers (K = 4096 / 11008, 16 stages) 557 -> 239 us; whole-step batches of
// four rows 387 -> 122 us (the same four layers, two launches) and 196 -> 139 us
// (154 TinyLlama linears).
#include <algorithm>
#include <type_traits>

#include "qxt_q4_0.h"

namespace qxt {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef unsigned int v2u __attribute__((ext_vector_type(2)));

constexpr int kMaxPasses = 4;    // chunks per wave and tile

// Most waves of a workgroup, by what a lane holds (registers).
template <int NB>
constexpr int kWaves = NB == 8 ? 8 : 16;

// RPL: rows per lane.  NB: blocks of a column per lane, 8 (a unit) or 4 (half
// a unit); the four lanes of a column hold a chunk.
template <int RPL, int NB>
struct RowsGeo {
    static constexpr int kRows = 4 * RPL;
    static constexpr int kChunk = 4 * NB;                           // blocks per wave step
    static constexpr int kUnits = NB / 2;                           // units of 8 blocks per wave step
    static constexpr int kPairs = kChunk / 2;                       // pairs of blocks per row and chunk
    static constexpr int kRowStep = 64 / kPairs;                    // rows a wave stages at once
    static constexpr int kWords = NB == 8 ? 36 : 20;                // weight words a lane loads
    static constexpr int kItems = (kRows + kRowStep - 1) / kRowStep;  // pairs of blocks staged per lane
    static constexpr int kPitch = kRows * 32 + 16;                  // bytes of a block's activation rows
    static constexpr int kScales = kChunk * kPitch;                 // then the scales: 64 floats per 4 blocks
    static constexpr int kChunkBytes = kScales + kChunk / 4 * 256;
    static size_t bytes(int chunks) { return static_cast<size_t>(chunks) * kChunkBytes + RPL * 256; }
};

// Native Q8_0 rows of one chunk: item k of a lane is blocks 2 p, 2 p + 1 of
// row kRowStep k + lane / kPairs, p = lane % kPairs (68 bytes, 4-byte aligned).
template <int RPL, int NB>
struct PairRegs {
    uint32_t d[RowsGeo<RPL, NB>::kItems][17];
};

template <int RPL, int NB>
__device__ __forceinline__ void load_pairs(const Q4Task &t, int r0, int m, int chunk, PairRegs<RPL, NB> &a) {
    using G = RowsGeo<RPL, NB>;
    const int lane = threadIdx.x & 63;
    const int pair = min(chunk * G::kPairs + lane % G::kPairs, t.blocks / 2 - 1);
#pragma unroll
    for (int k = 0; k < G::kItems; ++k) {
        const int r = r0 + min(G::kRowStep * k + lane / G::kPairs, m - 1);
        const uint8_t *p = t.act + r * t.act_stride + static_cast<size_t>(pair) * (2 * Q8_0_BYTES);
        typedef v4u v4u_a4 __attribute__((aligned(4)));
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const v4u x = global_in<v4u_a4>(p)[v];
#pragma unroll
            for (int j = 0; j < 4; ++j) a.d[k][4 * v + j] = x[j];
        }
        a.d[k][16] = global_in<uint32_t>(p)[16];
    }
}

// Their LDS image: per block and row the 32 bytes as four (word j, word j + 4)
// pairs, and the scales of blocks 4 q .. 4 q + 3 as 64 floats, lane
// (kg, 4 j + i) holding block 4 q + j of row kg + 4 i.
template <int RPL, int NB>
__device__ __forceinline__ void store_pairs(const PairRegs<RPL, NB> &a, uint8_t *s) {
    using G = RowsGeo<RPL, NB>;
    const int lane = threadIdx.x & 63;
    const int p = lane % G::kPairs;
    float *scales = reinterpret_cast<float *>(s + G::kScales);
#pragma unroll
    for (int k = 0; k < G::kItems; ++k) {
        const int r = G::kRowStep * k + lane / G::kPairs;
        if (G::kRows % G::kRowStep && r >= G::kRows) continue;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            uint32_t w[8];
#pragma unroll
            for (int j = 0; j < 8; ++j)
                w[j] = h ? a.d[k][9 + j] : __builtin_amdgcn_alignbyte(a.d[k][j + 1], a.d[k][j], 2);
            const int b = 2 * p + h;
            uint4 *dst = reinterpret_cast<uint4 *>(s + b * G::kPitch + r * 32);
            dst[0] = make_uint4(w[0], w[4], w[1], w[5]);
            dst[1] = make_uint4(w[2], w[6], w[3], w[7]);
            scales[(b >> 2) * 64 + (r & 3) * 16 + (b & 3) * 4 + (r >> 2)] =
                half_bits_to_float(h ? a.d[k][8] >> 16 : a.d[k][0] & 0xFFFFu);
        }
    }
}

// fp32 rows of one whole-unit chunk (four rows), quantised to Q8_0 here by the
// rule of q8_0_prepass_kernel: lane l holds half l % 2 of block l / 2 of every
// row, so that one exchange gives a block's maximum (the 4-element pieces of
// the other in-workgroup quantisers take three).
struct RowRegs {
    float4 v[4][4];
};

__device__ __forceinline__ void load_rows(const Q4Task &t, int m, int chunk, RowRegs &a) {
    const int lane = threadIdx.x & 63;
    const int b = min(chunk * 32 + (lane >> 1), t.blocks - 1);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const uint8_t *p = reinterpret_cast<const uint8_t *>(t.x) + min(r, m - 1) * t.x_stride +
                           static_cast<size_t>(b) * 128 + (lane & 1) * 64;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const v4u x = global_in<v4u>(p)[j];
            a.v[r][j] = make_float4(__uint_as_float(x[0]), __uint_as_float(x[1]), __uint_as_float(x[2]),
                                    __uint_as_float(x[3]));
        }
    }
}

__device__ __forceinline__ void store_rows(const RowRegs &a, uint8_t *s) {
    using G = RowsGeo<1, 8>;
    const int lane = threadIdx.x & 63;
    const int b = lane >> 1, h = lane & 1;
    float *scales = reinterpret_cast<float *>(s + G::kScales);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        float amax = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float4 &v = a.v[r][j];
            amax = fmaxf(fmaxf(fmaxf(amax, fabsf(v.x)), fmaxf(fabsf(v.y), fabsf(v.z))), fabsf(v.w));
        }
        amax = fmaxf(amax, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(amax), 0xB1, 0xF, 0xF, true)));
        float d, inv;
        q8_0_scale(amax, d, inv);
        uint8_t *dst = s + b * G::kPitch + r * 32 + h * 4;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float4 &v = a.v[r][j];
            *reinterpret_cast<uint32_t *>(dst + 8 * j) =
                pack_bytes(clamp127(rintf(v.x * inv)), clamp127(rintf(v.y * inv)), clamp127(rintf(v.z * inv)),
                           clamp127(rintf(v.w * inv)));
        }
        if (h == 0) scales[(b >> 2) * 64 + r * 16 + (b & 3) * 4] = half_bits_to_float(float_to_half_bits(d));
    }
}

// This lane's NB blocks of the chunk: a whole unit, or half h of one (bytes
// 72 h .. + 71).  Columns and units past the tile or K re-read the last one;
// their outputs are not stored, their terms not added.  The lane layout's
// 16-byte pieces straddle the halves: both halves load five and half 1 drops
// the first two words (lane_words).
template <int LAYOUT, int NB>
__device__ __forceinline__ void load_blocks(const Q4Task &t, int col, int unit, int h,
                                            uint32_t (&d)[RowsGeo<1, NB>::kWords]) {
    const int G = t.blocks >> 3;
    const int c = min(col, t.ncols - 1), g = min(unit, G - 1);
    if constexpr (LAYOUT == kLaneLayout) {
        const size_t u = static_cast<size_t>(t.wcol0 + c) * G + g;
        const QXT_GLOBAL v4u *src = global_in<v4u>(t.w + (u / kLaneGroup) * kGroupBytes + (u % kLaneGroup) * 16) +
                                    (NB == 4 ? 4 * h * kLaneGroup : 0);
#pragma unroll
        for (int v = 0; v < RowsGeo<1, NB>::kWords / 4; ++v) {
            const v4u x = src[v * kLaneGroup];
#pragma unroll
            for (int j = 0; j < 4; ++j) d[4 * v + j] = x[j];
        }
    } else {
        const uint8_t *p = t.w + static_cast<size_t>(t.wcol0 + c) * t.w_stride + static_cast<size_t>(g) * kUnitBytes +
                           (NB == 4 ? 72 * h : 0);
        typedef v4u v4u_a8 __attribute__((aligned(8)));
#pragma unroll
        for (int v = 0; v < (NB == 4 ? 4 : 9); ++v) {
            const v4u x = global_in<v4u_a8>(p)[v];
#pragma unroll
            for (int j = 0; j < 4; ++j) d[4 * v + j] = x[j];
        }
        if constexpr (NB == 4) {
            const v2u y = global_in<v2u>(p)[8];
            d[16] = y[0];
            d[17] = y[1];
        }
    }
}

// The lane's blocks at their places in a unit (the first half for NB = 4).
template <int LAYOUT, int NB>
__device__ __forceinline__ void lane_words(const uint32_t (&d)[RowsGeo<1, NB>::kWords], int h, uint32_t (&w)[36]) {
#pragma unroll
    for (int k = 0; k < (NB == 4 ? 18 : 36); ++k) {
        if constexpr (LAYOUT == kLaneLayout && NB == 4) w[k] = h ? d[k + 2] : d[k];
        else w[k] = d[k];
    }
}

__device__ __forceinline__ void swap16(uint32_t &a, uint32_t &b) {
    const v2u r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}
__device__ __forceinline__ void swap32(uint32_t &a, uint32_t &b) {
    const v2u r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}

// The block terms of one chunk: terms[i][b] of row kg + 4 i, column n.
template <int RPL, int NB>
__device__ __forceinline__ void chunk_terms(const uint32_t (&w)[36], const uint8_t *s,
                                            float (&terms)[RPL][4 * NB]) {
    using G = RowsGeo<RPL, NB>;
    const int lane = threadIdx.x & 63;
    const int kg = lane >> 4, slot = lane & 15;
    // Matrix row `slot` holds activation row slot / 4 + 4 (slot % 4); slots
    // past RPL re-read the first register's row (their outputs are unused).
    const int row = (slot >> 2) + 4 * ((slot & 3) < RPL ? (slot & 3) : 0);
    const uint8_t *arow = s + row * 32 + kg * 8;
    const float *scales = reinterpret_cast<const float *>(s + G::kScales) + lane;
    uint32_t words[4][NB], dw[4][NB];  // [lane group that held the block][its block]
    auto transpose = [&](auto ic) {
        constexpr int I = decltype(ic)::value;
        uint32_t sbits, q[4];
        unit_block<I>(w, sbits, q);
        swap16(q[0], q[1]);
        swap16(q[2], q[3]);
        swap32(q[0], q[2]);
        swap32(q[1], q[3]);
#pragma unroll
        for (int u = 0; u < 4; ++u) words[u][I] = q[u];
        uint32_t x = static_cast<uint32_t>(__float_as_int(half_bits_to_float(sbits) * 0.0625f)), y = x;
        swap16(x, y);
        uint32_t x2 = x, y2 = y;
        swap32(x, x2);
        swap32(y, y2);
        dw[0][I] = x;
        dw[1][I] = y;
        dw[2][I] = x2;
        dw[3][I] = y2;
    };
    transpose(std::integral_constant<int, 0>{});
    transpose(std::integral_constant<int, 1>{});
    transpose(std::integral_constant<int, 2>{});
    transpose(std::integral_constant<int, 3>{});
    if constexpr (NB == 8) {
        transpose(std::integral_constant<int, 4>{});
        transpose(std::integral_constant<int, 5>{});
        transpose(std::integral_constant<int, 6>{});
        transpose(std::integral_constant<int, 7>{});
    }
#pragma unroll
    for (int q = 0; q < NB; ++q) {
        const int das = __float_as_int(scales[q * 64]);
        auto block = [&](auto jc) {
            constexpr int j = decltype(jc)::value;
            const int b = 4 * q + j;
            const uint32_t x = words[b / NB][b % NB];
            const uint32_t lo = ((x << 4) & 0xF0F0F0F0u) ^ 0x80808080u, hi = (x & 0xF0F0F0F0u) ^ 0x80808080u;
            const long act = *reinterpret_cast<const long *>(arow + b * G::kPitch);
            const v4i zero = {0, 0, 0, 0};
            const v4i dot = __builtin_amdgcn_mfma_i32_16x16x32_i8(
                act, static_cast<long>((static_cast<uint64_t>(hi) << 32) | lo), zero, 0, 0, 0);
            const float dwf = __int_as_float(static_cast<int>(dw[b / NB][b % NB]));
            auto term = [&](auto ec) {
                constexpr int e = decltype(ec)::value;
                if constexpr (e < RPL)
                    terms[e][b] = (static_cast<float>(dot[e]) * dwf) *
                                  __int_as_float(__builtin_amdgcn_update_dpp(0, das, 0x150 + 4 * j + e, 0xF, 0xF, true));
            };
            term(std::integral_constant<int, 0>{});
            term(std::integral_constant<int, 1>{});
            term(std::integral_constant<int, 2>{});
            term(std::integral_constant<int, 3>{});
        };
        block(std::integral_constant<int, 0>{});
        block(std::integral_constant<int, 1>{});
        block(std::integral_constant<int, 2>{});
        block(std::integral_constant<int, 3>{});
    }
}

// Rows [r0, r0 + m) of columns [col_base, col_base + ncols) of one linear.
// X: the activation is fp32 rows (RPL = 1, NB = 8), else native Q8_0 rows.
// GROUPS: the workgroup may have more waves than K has chunks; each `chunks`
// of them are a group with a column tile of its own (waves past the last group
// only run the barriers).
template <int RPL, int LAYOUT, int NB, bool X = false, bool GROUPS = false>
__device__ __forceinline__ void rows_item(const Q4Task &t, int r0, int col_base, int ncols) {
    using G = RowsGeo<RPL, NB>;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int waves = static_cast<int>(blockDim.x >> 6);
    const int units = t.blocks >> 3;
    const int chunks = (units + G::kUnits - 1) / G::kUnits;
    const int half = (lane >> 4) & 1;
    const int passes = (chunks + waves - 1) / waves;
    const int groups = GROUPS ? max(1, waves / chunks) : 1;
    const int span = GROUPS ? min(waves, chunks) : waves;  // waves of a group
    const int group = GROUPS ? wave / span : 0;
    const int gwave = GROUPS ? wave - group * span : wave;  // this wave in its group
    const int m = min(t.rows - r0, G::kRows);
    float *run = reinterpret_cast<float *>(lds + static_cast<size_t>(chunks) * G::kChunkBytes) +
                 (GROUPS ? min(group, groups - 1) * (RPL * 64) : 0);

    // This wave stages chunks wave, wave + waves, ...; the first one's rows are
    // requested last, before the first tile's weights, and staged while those
    // are in flight.
    std::conditional_t<X, RowRegs, PairRegs<RPL, NB>> a;
    auto request = [&](int c) {
        if constexpr (X) load_rows(t, m, c, a);
        else load_pairs<RPL, NB>(t, r0, m, c, a);
    };
    auto stage = [&](int c) {
        uint8_t *s = lds + static_cast<size_t>(c) * G::kChunkBytes;
        if constexpr (X) store_rows(a, s);
        else store_pairs<RPL, NB>(a, s);
    };
    for (int p = passes - 1; p > 0; --p) {
        const int c = p * waves + wave;
        if (c >= chunks) continue;
        request(c);
        stage(c);
    }
    request(min(wave, chunks - 1));
    __builtin_amdgcn_sched_barrier(0);
    const int tiles = (ncols + 15) >> 4;
    const int steps = (tiles + groups - 1) / groups * passes;
    // Step q: column tile groups * (q / passes) + group, chunk (q % passes) *
    // span + gwave.
    int tile = group, pass = 0;
    auto load_step = [&](int tl, int ps, uint32_t (&d)[G::kWords]) {
        const int c = min(ps * span + gwave, chunks - 1);
        load_blocks<LAYOUT, NB>(t, col_base + min(tl, tiles - 1) * 16 + (lane & 15),
                                c * G::kUnits + (lane >> 4) * NB / 8, half, d);
    };
    uint32_t wr[G::kWords], wn[G::kWords];
    load_step(tile, 0, wr);
    __builtin_amdgcn_sched_barrier(0);
    if (wave < chunks) stage(wave);
    __syncthreads();

    auto step = [&](const uint32_t (&d)[G::kWords], uint32_t (&next)[G::kWords]) {
        const int nt = pass + 1 < passes ? tile : tile + groups, np = pass + 1 < passes ? pass + 1 : 0;
        load_step(nt, np, next);
        const int first = pass * span, mine = GROUPS && (group >= groups || tile >= tiles) ? chunks : first + gwave;
        float terms[RPL][G::kChunk];
        uint32_t w[36];
        lane_words<LAYOUT, NB>(d, half, w);
        if (mine < chunks) chunk_terms<RPL, NB>(w, lds + static_cast<size_t>(mine) * G::kChunkBytes, terms);
        // The waves add their terms in turn, in block order.
        const int active = min(span, chunks - first);
        for (int turn = 0; turn < active; ++turn) {
            if (GROUPS ? turn + first == mine : turn == wave) {
                float acc[RPL];
#pragma unroll
                for (int i = 0; i < RPL; ++i) acc[i] = mine == 0 ? 0.0f : run[i * 64 + lane];
#pragma unroll
                for (int u = 0; u < G::kUnits; ++u)
                    if (mine * G::kUnits + u < units)
#pragma unroll
                        for (int b = 8 * u; b < 8 * u + 8; ++b)
#pragma unroll
                            for (int i = 0; i < RPL; ++i) acc[i] = acc[i] + terms[i][b];
                if (mine + 1 < chunks) {
#pragma unroll
                    for (int i = 0; i < RPL; ++i) run[i * 64 + lane] = acc[i];
                } else {
                    const int col = tile * 16 + (lane & 15);
#pragma unroll
                    for (int i = 0; i < RPL; ++i) {
                        const int r = (lane >> 4) + 4 * i;
                        if (r < m && col < ncols)
                            global_out<float>(reinterpret_cast<uint8_t *>(t.y) +
                                              (r0 + r) * t.y_stride)[t.ocol0 + col_base + col] = acc[i];
                    }
                }
            }
            __syncthreads();
        }
        tile = nt;
        pass = np;
    };
    for (int q = 0;;) {
        step(wr, wn);
        if (++q >= steps) break;
        step(wn, wr);
        if (++q >= steps) break;
    }
}

template <int RPL, int LAYOUT, int NB>
__global__ __launch_bounds__(64 * kWaves<NB>) void q4_0_rows_kernel(Q4Task t) {
    const int col_base = static_cast<int>(blockIdx.x) * t.cpw;
    rows_item<RPL, LAYOUT, NB>(t, static_cast<int>(blockIdx.y) * RowsGeo<RPL, NB>::kRows, col_base,
                           min(t.cpw, t.ncols - col_base));
}

constexpr int kBatchBlocks = 8;  // NB of the batch kernels

template <int LAYOUT, int SOURCE, bool GROUPS>
__device__ __forceinline__ void rows_batch_item(const Q4Task &t, int col_base, int ncols) {
    auto run = [&](auto x) {
        constexpr bool X = decltype(x)::value;
        if (LAYOUT == kLaneLayout || (LAYOUT == kEitherLayout && t.lanes))
            rows_item<1, kLaneLayout, kBatchBlocks, X, GROUPS>(t, 0, col_base, ncols);
        else
            rows_item<1, kNativeRows, kBatchBlocks, X, GROUPS>(t, 0, col_base, ncols);
    };
    if (SOURCE == kRowsFp32 || (SOURCE == kRowsEither && t.x != nullptr)) run(std::true_type{});
    else run(std::false_type{});
}

template <int LAYOUT, int SOURCE, bool GROUPS>
__global__ __launch_bounds__(64 * kWaves<kBatchBlocks>) void q4_0_rows_batch_kernel(const Q4Task *__restrict__ tasks,
                                                                                    const Q4Item *__restrict__ items) {
    const Q4Item item = items[blockIdx.x];
    rows_batch_item<LAYOUT, SOURCE, GROUPS>(tasks[item.task], item.col_base, item.ncols);
}

template <int LAYOUT, int SOURCE, bool GROUPS>
__global__ __launch_bounds__(64 * kWaves<kBatchBlocks>) void q4_0_rows_arg_batch_kernel(Q4ArgBatch a) {
    const int i = static_cast<int>(blockIdx.x);
    int ti = 0;
#pragma unroll
    for (int j = 1; j < kArgTasks; ++j) ti += i >= a.first_item[j] ? 1 : 0;
    const Q4Task t = a.task[ti];
    const int col_base = (i - a.first_item[ti]) * t.cpw;
    rows_batch_item<LAYOUT, SOURCE, GROUPS>(t, col_base, min(t.cpw, t.ncols - col_base));
}

template <int NB>
int chunks_of(int blocks) {
    return (blocks / 8 + NB / 2 - 1) / (NB / 2);
}

template <int RPL, int NB>
int launch_rows(Q4Task t, hipStream_t stream) {
    const int chunks = chunks_of<NB>(t.blocks);
    const int waves = rows_waves(chunks, kWaves<NB>);
    const int groups = (t.rows + 4 * RPL - 1) / (4 * RPL);
    const size_t lds = RowsGeo<RPL, NB>::bytes(chunks);
    t.cpw = 16 * rows_steps(static_cast<long>(groups) * ((t.ncols + 15) / 16),
                            compute_units() * rows_resident(waves, NB == 8 ? kRowsWavesPerCu : 16, lds));
    const dim3 grid((t.ncols + t.cpw - 1) / t.cpw, groups, 1);
    return t.lanes ? launch("q4_0_linear_kernel", q4_0_rows_kernel<RPL, kLaneLayout, NB>, grid, dim3(64 * waves), lds,
                            stream, t)
                   : launch("q4_0_linear_kernel", q4_0_rows_kernel<RPL, kNativeRows, NB>, grid, dim3(64 * waves), lds,
                            stream, t);
}

template <int RPL, int NB>
bool fits(int blocks) {
    const int chunks = chunks_of<NB>(blocks);
    return chunks <= kWaves<NB> * kMaxPasses && RowsGeo<RPL, NB>::bytes(chunks) <= kRowsLds;
}

// The LDS of both chunk sizes, so that a shape fits or not by its rows and K.
template <int RPL>
bool fits(int blocks) {
    return fits<RPL, 4>(blocks) && fits<RPL, 8>(blocks);
}

bool fits(int blocks, int rows_per_lane) {
    return rows_per_lane == 1   ? fits<1>(blocks)
           : rows_per_lane == 2 ? fits<2>(blocks)
           : rows_per_lane == 3 ? fits<3>(blocks)
                                : fits<4>(blocks);
}

// Whole units, 16-byte aligned weight rows, 4-byte aligned Q8_0 rows.
bool layout_ok(const Q4Task &t) {
    return t.blocks % 8 == 0 && aligned(t.w, 16) && t.w_stride % 16 == 0 && t.x == nullptr && aligned(t.act, 4) &&
           t.act_stride % 4 == 0;
}

}  // namespace

// Sixteen or more native rows: row groups of this kernel against the 64 x 64
// prefill tiles (qxt_q4_0_tiled.hip), whose time is the K of one tile until
// their grid fills the chip.  Both from sweeps on MI355X (us): this kernel 2.5 +
// 3.6 ns per tile, group and 32 blocks (1.7 times that where one workgroup's LDS
// takes a CU: more than 8 rows past K = 4096); the tiles 2.5 + 7.2 per 1024 of K,
// from 300 workgroups 0.024 each.  Measured, tiles -> this kernel: 16 rows
// 5632 x 2048 40.9 -> 7.2, 64 rows 41.3 -> 14.3, 128 rows 41.2 -> 34.2; 64 rows
// 2048 x 5632 18.2 -> 12.6, 96 rows 18.1 -> 18.7 (not taken); 24 rows 4096 x 11008
// 36.8 -> 24.9; 16 rows 2048 x 32000 24.0 -> 16.4, 24 rows 23.8 -> 31.2 (not taken).
static bool takes_native_prefill(const Q4Task &t, long tiles) {
    const int rpl = fits(t.blocks, 4) ? 4 : 2;
    const double groups = (t.rows + 4 * rpl - 1) / (4 * rpl), chunks = (t.blocks + 31) / 32;
    const double here = 2.5 + 3.6e-3 * (rpl == 4 && t.blocks > 128 ? 1.7 : 1.0) * tiles * groups * chunks;
    const double workgroups = static_cast<double>((t.rows + 63) / 64) * ((t.ncols + 63) / 64);
    return 1.1 * here < 2.5 + t.blocks / 32.0 * std::max(7.2, 0.024 * workgroups);
}

int q4_0_rows_linear(const Q4Task &t, hipStream_t stream) {
    if (t.rows < 2 || !layout_ok(t)) return QXT_CAPABILITY_MISSING;
    const long tiles = (t.ncols + 15) / 16, cus = compute_units();
    const bool taken = t.rows < 16 ? rows_linear_takes(t.lanes != 0, t.rows, t.blocks, tiles, cus)
                       : t.lanes   ? rows_lanes_prefill_takes(t.rows, t.blocks, tiles, cus)
                                   : takes_native_prefill(t, tiles);
    if (!taken) return QXT_CAPABILITY_MISSING;
    // The fewest rows per lane that leave every workgroup a CU of its own;
    // larger grids take all rows at once (K = 5632, N = 2048, 5 rows: two row
    // groups 6.4 us, one 7.0; K = 2048, N = 5632: 6.6 and 5.3).
    int rpl = 0;
    for (int r = 1; r <= 4 && rpl == 0; ++r)
        if (fits(t.blocks, r) && (tiles * ((t.rows + 4 * r - 1) / (4 * r)) <= cus || 4 * r >= t.rows)) rpl = r;
    if (rpl == 0) rpl = fits(t.blocks, 4) ? 4 : fits(t.blocks, 2) ? 2 : 1;
    if (!fits(t.blocks, rpl)) return QXT_CAPABILITY_MISSING;
    const long groups = (t.rows + 4 * rpl - 1) / (4 * rpl);
    // Half-unit chunks while the grid is latency-bound: half the instructions
    // per wave, twice the turns (native rows, 8 rows, us, half / whole units:
    // K = 2048, N = 5632 5.6 / 6.2; K = 11008, N = 4096 13.1 / 14.1; K = 4096,
    // N = 11008 13.8 / 12.7.  Lane layout past K = 2048: its 16-byte pieces
    // straddle the halves, 15.6 / 14.6 at K = 11008, N = 4096).
    const bool small = tiles * groups <= 2 * cus && (!t.lanes || t.blocks <= 64);
    switch (rpl) {
        case 1: return small ? launch_rows<1, 4>(t, stream) : launch_rows<1, 8>(t, stream);
        case 2: return small ? launch_rows<2, 4>(t, stream) : launch_rows<2, 8>(t, stream);
        case 3: return small ? launch_rows<3, 4>(t, stream) : launch_rows<3, 8>(t, stream);
        default: return small ? launch_rows<4, 4>(t, stream) : launch_rows<4, 8>(t, stream);
    }
}

static_assert(RowsGeo<1, kBatchBlocks>::kChunkBytes == kRowsChunkBytes && kWaves<kBatchBlocks> == kRowsWaves &&
                  kMaxPasses == kRowsMaxPasses,
              "the plan's figures of a chunk and a workgroup");

static RowsTiles tiles_by_chunks(const Q4Task *tasks, uint32_t count) {
    RowsTiles tiles;
    for (uint32_t i = 0; i < count; ++i)
        tiles[chunks_of<kBatchBlocks>(tasks[i].blocks)] += (static_cast<long>(tasks[i].ncols) + 15) / 16;
    return tiles;
}

bool q4_0_rows_batch_takes(const Q4Task *tasks, uint32_t count) {
    double units = 0.0, columns = 0.0;
    bool fp32 = false;
    for (uint32_t i = 0; i < count; ++i) {
        Q4Task t = tasks[i];
        fp32 = fp32 || t.x != nullptr;
        t.x = nullptr;
        if (t.rows > 4 || !layout_ok(t) || !fits(t.blocks, 1)) return false;
        units += t.blocks / 8.0 * t.ncols;
        columns += t.ncols;
    }
    if (columns > 16.0 * (1 << 24)) return false;  // a table of one item per 16 columns
    return rows_batch_preferred(tiles_by_chunks(tasks, count), units, fp32, compute_units());
}

RowsPlan q4_0_rows_plan(Q4Task *tasks, uint32_t count) {
    const RowsPlan plan = rows_batch_plan(tiles_by_chunks(tasks, count), compute_units());
    for (uint32_t i = 0; i < count; ++i)
        tasks[i].cpw = std::min(plan.columns(chunks_of<kBatchBlocks>(tasks[i].blocks)), (tasks[i].ncols + 15) / 16 * 16);
    return plan;
}

namespace {

// Mixed sources have one instantiation for every layout.
template <int SOURCE, bool GROUPS>
int launch_batch(const Q4ArgBatch *args, const Q4Task *tasks, const Q4Item *items, uint32_t grid, const RowsPlan &plan,
                 int layout, hipStream_t stream) {
    const dim3 blocks(grid), threads(64 * plan.waves);
    auto run = [&](auto lc) {
        constexpr int L = decltype(lc)::value;
        return args != nullptr ? launch("q4_0_batch_kernel", q4_0_rows_arg_batch_kernel<L, SOURCE, GROUPS>, blocks,
                                        threads, plan.lds, stream, *args)
                               : launch("q4_0_batch_kernel", q4_0_rows_batch_kernel<L, SOURCE, GROUPS>, blocks, threads,
                                        plan.lds, stream, tasks, items);
    };
    if constexpr (SOURCE != kRowsEither) {
        if (layout == kLaneLayout) return run(std::integral_constant<int, kLaneLayout>{});
        if (layout == kNativeRows) return run(std::integral_constant<int, kNativeRows>{});
    }
    return run(std::integral_constant<int, kEitherLayout>{});
}

template <bool GROUPS>
int launch_batch(const Q4ArgBatch *args, const Q4Task *tasks, const Q4Item *items, uint32_t grid, const RowsPlan &plan,
                 int layout, RowsSource source, hipStream_t stream) {
    return source == kRowsQ8 ? launch_batch<kRowsQ8, GROUPS>(args, tasks, items, grid, plan, layout, stream)
           : source == kRowsFp32
               ? launch_batch<kRowsFp32, GROUPS>(args, tasks, items, grid, plan, layout, stream)
               : launch_batch<kRowsEither, GROUPS>(args, tasks, items, grid, plan, layout, stream);
}

}  // namespace

int q4_0_rows_batch(const Q4ArgBatch *args, const Q4Task *tasks, const Q4Item *items, uint32_t grid,
                    const RowsPlan &plan, int layout, RowsSource source, hipStream_t stream) {
    return plan.groups ? launch_batch<true>(args, tasks, items, grid, plan, layout, source, stream)
                       : launch_batch<false>(args, tasks, items, grid, plan, layout, source, stream);
}

}  // namespace qxt
