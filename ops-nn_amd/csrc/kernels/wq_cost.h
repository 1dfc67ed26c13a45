// What the weight-only kernels take, in microseconds: the estimates that the dispatch of wq_nk.hip, wq_dense.hip and wq_wide.hip compares
// where two kernels can run a call.  First those of wq_nk.hip and wq_dense.hip:  Fitted to measured times of 513 calls of 1 .. 64 rows and 368 of 65 .. 2100 (weights cold, K 1024 ..
// 14336, N 1024 .. 28680); profiles/weight_only_routes.txt has both sides' times.  Shapes and types only, so that both phases of a
// call agree.
#pragma once
#include <cmath>

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
// For the rule of wq_wide.hip, of both sides: what a call typically takes, the geometric mean of its time with the weight from memory and
// from the last-level cache.  Fitted to 3800 calls (M 1 .. 512, K 1024 .. 18432, N 1024 .. 28672, both storages, groups of 32 to K) that were
// timed on either side in both states; median error 2 to 6 %, by kernel.  Next to each kernel's plan where it has one.
inline double wq_typical_turns(int64_t wgs, double two)   // workgroups one after the other, two at a time on a CU
{
    return wgs <= 256 ? 1.0 : wgs <= 512 ? two : two * 0.5 * ((double)wgs / 512.0 + (double)((wgs + 511) / 512));
}
inline double wq_typical_both(double cu, double hbm) { return std::cbrt(cu * cu * cu + hbm * hbm * hbm); }
inline double wq_typical_mb(int wbits, int64_t N, int64_t K) { return (double)N * (double)K * (double)wbits / 8e6; }
// One pass of the streaming kernel.  Up to 16 rows its four waves share K against a narrow N.
inline double wq_stream_typical_us(const OpsnnWqmmArgs& a, const WqForm& f)
{
    const int w8 = f.wbits == 8, bf = a.x_dtype == DT_BF16;
    const bool off = a.offset != nullptr;
    if (a.M > 16) {
        static const double rate[2][2] = {{1.0, 0.99}, {0.98, 0.86}}, offs[2][2] = {{0.059, 0.224}, {0.049, 0.176}};
        return wq_stream_pass_us(f.wbits, bf, a.M, a.N, a.K) * rate[w8][bf] * (off ? 1.0 + offs[w8][bf] : 1.0) - 0.3 + 1.83e-6 * (double)a.M * (double)a.N;
    }
    static const double rate[2][2] = {{1.87, 2.78}, {2.36, 3.29}}, offs[2][2] = {{0.2, 0.61}, {0.23, 0.35}};
    const int64_t chunks = a.K / (w8 ? 64 : 128), blocks = (a.N + 15) / 16;
    const bool share_k = blocks < 1024 && chunks % 4 == 0 && chunks >= 8;
    double share = blocks <= 1024 ? 1.0 : blocks <= 2048 ? 1.92 : 1.92 * (double)blocks / 2048.0;
    if (share_k) share = 0.37 * (blocks > 224 ? 1.14 * (double)blocks / 256.0 : 1.0);
    return 5.47 + (double)a.K / 1024.0 * rate[w8][bf] * (off ? 1.0 + offs[w8][bf] : 1.0) * share;
}
inline double wq_general_typical_us(const OpsnnWqmmArgs& a)
{
    return 1.1 + wq_general_pass_us(a.M, a.N, a.K) * (a.offset ? 0.915 : 0.871) + 0.85e-6 * (double)a.M * (double)a.N;
}
// The kernel that holds x whole in LDS, its four waves a quarter of K each.
inline double wq_resx_typical_us(const OpsnnWqmmArgs& a, const WqForm& f)
{
    static const double rate[2][2] = {{0.365, 0.74}, {0.55, 0.876}};
    const double w = (double)((a.N + 15) / 16) / 256.0, share = w <= 1.0 ? 1.0 : w <= 2.0 ? 1.67 : 0.84 * w;
    const double cu = share * (double)a.K / 1024.0 * (rate[f.wbits == 8][a.x_dtype == DT_BF16] + (a.offset ? 0.283 : 0.0));
    return 3.97 + 1.02e-4 * (double)a.M * (double)a.K + wq_typical_both(cu, wq_typical_mb(f.wbits, a.N, a.K) / 5.06);
}
// The x-in-registers kernel with K in segments (median error 7 %).
inline double wq_xreg_typical_us(const OpsnnWqmmArgs& a, const WqForm& f, const WqXregPlan& x)
{
    static const double rate[2][2] = {{0.55, 1.01}, {0.0, 0.18}};
    const int64_t cus = (256 + x.splits - 1) / x.splits, rounds = ((a.N + 15) / 16 + cus - 1) / cus;
    const double piece = rate[f.wbits == 8][a.x_dtype == DT_BF16] + (a.offset ? 0.52 : 0.0), held = (double)(x.nw * x.nch);
    const double out_m = (double)a.M * (double)a.N * (a.N % 4 ? 2e-6 : 1e-6);
    return 3.12 + 3.28 * held / 64.0 + wq_typical_both((double)rounds * held / 16.0 * piece, wq_typical_mb(f.wbits, a.N, a.K) / 5.18) +
           (x.splits > 1 ? 3.01 + 5.99 * (double)x.splits * out_m : 0.0);
}
// What dequantising 4096 k of a workgroup's columns takes in the many-rows kernel.
inline double wq_rows_dequant_us(int wbits, bool bf16) { return wbits == 4 ? (bf16 ? 8.0 : 1.7) : (bf16 ? 16.2 : 9.2); }

}  // namespace opsnn
