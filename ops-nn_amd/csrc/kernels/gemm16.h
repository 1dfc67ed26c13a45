// 16-bit operand GEMM (gemm16.hip): the dense step behind a pass that has widened quantized operands to fp16 / bf16.
#pragma once
#include "launch.h"
#include "qgemm_core.hip.h"

namespace opsnn {

// How a [M, K] x [N, K] product of 16-bit operands is tiled.  cfg: 8 .. 11 the four-wave kernel with 256 x 32*cfg tiles
// (qmm_int8_wide.hip), else the OPSNN_VARIANT_I8_* tile of that number.  splits > 1: K split over workgroups, fp32 partial sums
// [splits][M][N].  rows or cols: only so many of the first rows or columns that way, in a launch of its own, the others with rest_cfg and
// rest_splits in a second one.  us: the estimate that the choice rests on.
struct Gemm16Plan {
    int cfg = OPSNN_VARIANT_I8_128, splits = 1;
    double us = 0;
    int64_t rows = 0, cols = 0;
    int rest_cfg = OPSNN_VARIANT_I8_128, rest_splits = 1;
};
Gemm16Plan gemm16_plan(int64_t M, int64_t N, int64_t K);
inline uint64_t gemm16_part_bytes(const Gemm16Plan& pl, int64_t M, int64_t N)
{
    const int splits = pl.rows || pl.cols ? pl.rest_splits : pl.splits;   // (of two launches only the second one splits K)
    return splits > 1 ? ((uint64_t)splits * (uint64_t)(M - pl.rows) * (uint64_t)(N - pl.cols) * 4 + 255) / 256 * 256 : 0;
}
// p: a / b with strides in bytes, KB = 2 K, K % 64 == 0, out [M, N] of the operands' type with row pitch ldc, a floating bias (may be
// null).  `part`: gemm16_part_bytes of the plan.
int launch_gemm16(QgemmParams p, const Gemm16Plan& pl, bool bf16, float* part, hipStream_t st);

}  // namespace opsnn
