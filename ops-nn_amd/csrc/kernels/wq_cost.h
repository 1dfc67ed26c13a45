// What the weight-only kernels take, in microseconds: the estimates that the dispatch of wq_nk.hip and wq_dense.hip compares where
// two kernels can run a call.  Fitted to measured times of 513 calls of 1 .. 64 rows and 368 of 65 .. 2100 (weights cold, K 1024 ..
// 14336, N 1024 .. 28680); profiles/weight_only_routes.txt has both sides' times.  Shapes and types only, so that both phases of a
// call agree.
#pragma once
#include "common.hip.h"
#include "launch.h"

namespace opsnn {

// A weight-only call's form: what the kernels' conditions look at.
struct WqForm {
    int wbits;
    bool nk, stream, rows;   // K-contiguous; whole chunks and groups of a power of two of them (wqmm_stream.hip.h); the many-rows kernel's shapes
    int64_t group;           // K without groups
};
inline WqForm wq_form(const OpsnnWqmmArgs& a)
{
    WqForm f;
    f.wbits = a.w_dtype == DT_I4 ? 4 : 8;
    f.nk = a.w.row_stride == 1 && a.w.col_stride == a.K;
    f.group = a.group > 0 && a.group < a.K ? a.group : a.K;
    const int64_t kc = 4 * (128 / f.wbits), cpg = f.group < a.K ? f.group / kc : 1;
    f.stream = a.K % kc == 0 && (f.group >= a.K || (f.group % kc == 0 && (cpg & (cpg - 1)) == 0));
    f.rows = f.stream && a.N % 32 == 0 && a.N >= 256 && a.K % (2 * kc) == 0;
    return f;
}

// One pass of the streaming kernel (wqmm_stream.hip.h) over the weight: up to 64 rows, workgroups of 64 columns, two of which a CU
// can hold (median error 4 %).
inline double wq_stream_pass_us(int wbits, bool bf16, int64_t rows, int64_t N, int64_t K)
{
    const double wgs = (double)((N + 63) / 64), share = wgs <= 256.0 ? 1.0 : wgs <= 512.0 ? 1.53 : 1.53 * wgs / 512.0;
    const double per = rows <= 32 ? (2.47 + 0.027 * (double)rows) * (bf16 ? 1.38 : 1.0) : (3.3 + 0.035 * (double)rows) * (bf16 ? 1.19 : 1.0);
    return 4.6 + (double)K / 1024.0 * per * share * (wbits == 8 ? 1.3 : 1.0);
}
// One pass of the general kernel (wqmm.hip) in its best form, fp16 with 4-bit weights (median error 4 %); with bf16 or 8-bit weights it
// takes 1.2 to 4 times as long and is never the faster one.  From 2048 k against fewer than 1024 column blocks its waves share K.
inline double wq_general_pass_us(int64_t rows, int64_t N, int64_t K)
{
    const int i = rows <= 16 ? 0 : rows <= 32 ? 1 : 2;
    const double blocks = (double)((N + 15) / 16);
    if (blocks < 1024.0 && K >= 2048) {
        static const double t[3] = {9.0, 11.8, 19.3};
        const double share = 0.86 * blocks / 256.0;
        return 2.6 + (double)K / 4096.0 * t[i] * (share > 1.0 ? share : 1.0);
    }
    static const double t[3] = {5.9, 6.9, 9.0};
    const double wgs = (double)((N + 63) / 64), two = K % 2048 == 0 ? 1.58 : 1.28;   // (rows at a power-of-two pitch share fewer channels)
    return 2.6 + (double)K / 1024.0 * t[i] * (wgs <= 256.0 ? 1.0 : wgs <= 512.0 ? two : two * wgs / 512.0);
}
inline bool wq_general_counts(const OpsnnWqmmArgs& a, const WqForm& f) { return f.wbits == 4 && a.x_dtype == DT_F16 && f.group % 64 == 0 && a.K % 32 == 0; }
template <typename PASS>
inline double wq_passes_of_64_us(int64_t M, PASS&& pass)
{
    double us = 0.0;
    for (int64_t m0 = 0; m0 < M; m0 += 64) us += pass(M - m0 < 64 ? M - m0 : 64);
    return us;
}
// What dequantising 4096 k of a workgroup's columns takes in the many-rows kernel.
inline double wq_rows_dequant_us(int wbits, bool bf16) { return wbits == 4 ? (bf16 ? 8.0 : 1.7) : (bf16 ? 16.2 : 9.2); }

}  // namespace opsnn
