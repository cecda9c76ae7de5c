// The decode GEMV's second stage for a few batch rows (nq_gemv_split.hip): plan and launch.
#pragma once

#include "nq_common.h"

namespace nq {

// One stage 2: y = sat(s_out * U z), z = z_hi + z_lo [batch][zpitch] with zeros past the rank.
struct SplitItem {
    const uint32_t* u_bits;  // [m][wr], 16-byte aligned
    const uint16_t* s_out;
    uint16_t* y;
    const uint16_t* resid;  // residual epilogue: laid out as y
    const uint16_t* z_hi;   // 16-byte aligned, zpitch a multiple of 8
    const uint16_t* z_lo;
    int m, wr, zpitch;
    int ystride;  // elements between batch rows of y and resid
    int blocks;   // set by the launch
    int vec4;     // set by the launch
};

constexpr int kSplitItems = 4;
constexpr int kSplitMaxBatch = 32;  // the ranges that split_plan was measured on
constexpr int kSplitMaxWords = 144;
struct SplitTable {
    SplitItem item[kSplitItems];
    int count;
};

enum SplitEpilogue { kSplitStore = 0, kSplitResidual = 1, kSplitGated = 2 };

// Block shape: 16 * row_tiles rows of U by 8 * col_tiles batch rows, the k range shared by `waves` waves.
struct SplitPlan {
    int row_tiles, col_tiles, waves;
};

// The block shape for one item (or a gated pair) of m rows and wr words.
SplitPlan split_plan(int batch, int m, int wr);

// One launch over the table's items (kSplitGated: the pair). dtype: NQ_F16 or NQ_BF16.
int launch_split(int dtype, SplitTable& tab, int batch, SplitEpilogue epi, const SplitPlan& p, hipStream_t st);

}  // namespace nq
