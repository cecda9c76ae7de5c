// The decode GEMV's stages for many batch rows (nq_gemv_rows.hip): plan and launches.
#pragma once

#include "nq_common.h"

namespace nq {

// One stage over many batch rows. Stage 1 (z = V (s_in * x) * s_mid): x [batch][K] in T, words of V
// [rows][wpr], scale s_mid (or nullptr), the intermediate written as z_hi + z_lo. Stage 2 (y = s_out *
// U z): the operands are z_hi and z_lo [batch][zpitch], words of U, scale s_out, y written.
struct RowsArgs {
    const uint32_t* words;
    const uint16_t* x;      // stage 1
    const uint16_t* s_in;   // stage 1
    const uint16_t* scale;  // per feature: s_mid or nullptr, s_out
    uint16_t* z_hi;
    uint16_t* z_lo;
    uint16_t* y;            // stage 2
    float* part;            // stage 1 over several k ranges: [splits][batch][kpad] raw sums
    int rows, wpr, batch;   // features (r, m), words per feature, batch rows
    int K;                  // stage 1: columns of x (n); stage 2: columns of z that are multiplied
    int kpad, zpitch;       // stage 1 output: columns [rows, kpad) and [kpad, zpitch) get zeros
};

// Features of a block (by 64 batch rows; kRows256q32: by 32), and the wave groups its k steps are shared by.
enum RowsTile { kRows256, kRows128x2, kRows128x4, kRows256q32 };

struct RowsPlan {
    RowsTile tile;
    int splits, split_steps;  // k ranges of split_steps 64-k steps (stage 1)
    size_t part_bytes;
};

// Whether, and how, stage 1 / stage 2 runs these kernels (part_room: bytes of workspace for the raw
// sums of several k ranges).
bool rows_stage1_plan(int64_t batch, int64_t n, int64_t r, int64_t kpad, size_t part_room, RowsPlan& p);
bool rows_stage2_plan(int64_t batch, int64_t m, int64_t wr, RowsPlan& p);

// dtype: NQ_F16 or NQ_BF16. With p.splits > 1 stage 1 leaves raw sums in a.part.
void launch_rows_stage1(int dtype, const RowsArgs& a, const RowsPlan& p, hipStream_t st);
void launch_rows_stage2(int dtype, const RowsArgs& a, const RowsPlan& p, hipStream_t st);

}  // namespace nq
