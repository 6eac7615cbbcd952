// The int4 LM head of a few rows with what stands around it (int4_head.hip).
#pragma once
#include <algorithm>

#include "linear_common.h"

constexpr int kHeadRowsLds = 156 * 1024;  // of a CU's 160 KiB

// Two to sixteen rows x [rows][K], normalised first where gamma is given -> y [rows][N]; with idx_out the arg-max of every row over its first `cols` columns, and with
// adv.cur_tok the winners fed back as the next tokens and the counters moved on.
bool agpu_int4_head_rows_supported(const agpu_ctx *ctx, const float *x, int rows, int N, int K, int group);
int32_t agpu_int4_head_rows_launch(agpu_ctx *ctx, const float *x, const float *gamma, const float *beta, float eps, const uint32_t *packed, const float *scales, float *y, int rows,
                                   int N, int K, int group, int cols, uint32_t *idx_out, int last, const ArgmaxAdvance &adv);
