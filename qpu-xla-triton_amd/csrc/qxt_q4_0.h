// Task description and device helpers shared by the small-M Q4_0 kernels
// (qxt_q4_0.hip, qxt_q4_0_rows.hip).
#pragma once

#include "qxt_common.h"
#include "qxt_q4_0_rows_plan.h"

namespace qxt {

struct Q4Task {
    const float *x;        // fp32 rows quantised to Q8_0 in the workgroup, or nullptr
    size_t x_stride;
    const uint8_t *act;    // native Q8_0 blocks [rows, blocks, 34] (when x is nullptr)
    const uint8_t *w;      // Q4_0 blocks [N, blocks, 18]
    float *y;              // fp32 output
    int32_t *dots;         // debug: int32 block dots [rows, ncols, blocks]
    size_t act_stride, w_stride, y_stride;  // row strides in bytes
    int rows, blocks, wcol0, ocol0, ncols, cpw;
    int lanes;             // weight in the lane-interleaved layout (w = packed matrix base)
};

constexpr int kLaneGroup = 64;                      // units per lane group
constexpr int kUnitBytes = 144;                     // 8 Q4_0 blocks of one column
constexpr int kGroupBytes = kLaneGroup * kUnitBytes;  // 9216

struct Q4Item {
    int task;
    int col_base;
    int ncols;  // columns of this work item (<= the task's cpw)
};

typedef unsigned int v4u __attribute__((ext_vector_type(4)));

// Batch kernels read their tensor pointers from a device table, so the
// compiler cannot tell they address global memory and would emit FLAT
// loads.  A FLAT load also counts against the LDS counter, which turns every
// later wait for an LDS access into a wait for all outstanding weight loads
// (activation staging then starts only after the weights have landed).
// Every tensor access goes through a global-address-space pointer instead.
#define QXT_GLOBAL __attribute__((address_space(1)))
template <typename T>
__device__ __forceinline__ const QXT_GLOBAL T *global_in(const void *p) {
    return (const QXT_GLOBAL T *)p;
}
template <typename T>
__device__ __forceinline__ QXT_GLOBAL T *global_out(void *p) {
    return (QXT_GLOBAL T *)p;
}
// Block i (0..7) of a 144-byte unit held as 36 little-endian words: returns
// the fp16 scale bits and the 4 words of packed nibbles.
template <int I>
__device__ __forceinline__ void unit_block(const uint32_t (&d)[36], uint32_t &sbits, uint32_t (&qs)[4]) {
    if constexpr ((I & 1) == 0) {
        constexpr int k = 9 * I / 2;  // block starts word-aligned: d then nibbles at +2 bytes
        sbits = d[k] & 0xFFFFu;
#pragma unroll
        for (int t = 0; t < 4; ++t) qs[t] = __builtin_amdgcn_alignbyte(d[k + t + 1], d[k + t], 2);
    } else {
        constexpr int k = (9 * I - 1) / 2;  // block starts at a half word: nibbles word-aligned
        sbits = d[k] >> 16;
#pragma unroll
        for (int t = 0; t < 4; ++t) qs[t] = d[k + 1 + t];
    }
}

// Weight layout of a kernel instantiation: native rows, lane layout, or
// either (read from the task).  Separate instantiations keep the lane
// layout's non-temporal loads from being merged with the native rows'
// ordinary loads of the other branch.
enum WeightLayout { kNativeRows = 0, kLaneLayout = 1, kEitherLayout = 2 };

// A batch of at most kArgTasks tasks travels in the kernel arguments: each
// workgroup finds its task and column tile from its index, without the two
// dependent reads of a device table (item, then task) before its first
// weight or activation request.  Task j's items start at first_item[j]
// (INT_MAX past the last task) and are its column tiles of cpw columns in
// order.
constexpr int kArgTasks = 4;
struct Q4ArgBatch {
    int first_item[kArgTasks];
    Q4Task task[kArgTasks];
};

// Two or more rows on 16 x 16 matrix-core tiles (qxt_q4_0_rows.hip).  The
// single linear returns QXT_CAPABILITY_MISSING (no message, nothing launched)
// for shapes it does not take.  The batch takes tasks of at most four rows each,
// planned by q4_0_rows_plan (which sets every task's cpw), whose activations are
// `source`; `args` or, when that is null, the device tables `tasks` and `items`.
enum RowsSource { kRowsQ8 = 0, kRowsFp32 = 1, kRowsEither = 2 };  // kRowsEither: fp32 where the task's x is set
int q4_0_rows_linear(const Q4Task &t, hipStream_t stream);
bool q4_0_rows_batch_takes(const Q4Task *tasks, uint32_t count);
RowsPlan q4_0_rows_plan(Q4Task *tasks, uint32_t count);
int q4_0_rows_batch(const Q4ArgBatch *args, const Q4Task *tasks, const Q4Item *items, uint32_t grid,
                    const RowsPlan &plan, int layout, RowsSource source, hipStream_t stream);

}  // namespace qxt
