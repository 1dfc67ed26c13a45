// Dense product of two 16-bit operands (fp16 or bf16, both K-contiguous) with fp32 sums, a bias in the epilogue and an output of
// the operands' type: the step behind the pass that dequantises a weight once per call (wq_dense.hip).  The kernels
// are the tile kernels of the quantized modes with another matrix instruction: everything in them is addressed in bytes
// of K, and a lane's 16 bytes feed one 16-bit instruction where they feed one int8 instruction.
#include "gemm16.h"
#include "launch.h"

namespace opsnn {

int launch_16_wide(const QgemmParams& p, int fn, bool bf16, hipStream_t st);   // qmm_int8_wide.hip

// out[m, n] = rounded(sum over the splits, in split order, + bias[n])
template <int W>
__global__ __launch_bounds__(256) void gemm16_splitk_reduce_kernel(QgemmParams p, int out_dt)
{
    splitk_rows<W>((const float*)p.part, p.splits, p.M * p.N, p.M, p.N, [&](int64_t m, int64_t n0, float (&v)[W]) {
        if (p.bias) {
#pragma unroll
            for (int e = 0; e < W; e++) v[e] = v[e] + load_scalar_as_f32(p.bias, p.bias_dt, n0 + e);
        }
        store_cols(p.out, out_dt, m * p.ldc + n0, v);
    });
}

template <int MODE, int BM, int BN, int WGM, int WGN, int STAGES>
static int launch_split16(const QgemmParams& p, hipStream_t st)
{
    constexpr int BK = 128;
    if (!p.part || p.splits < 2 || (p.KB % BK) != 0 || p.splits > p.KB / BK / 2) return -1;
    const int tiles_m = (int)((p.M + BM - 1) / BM), tiles_n = (int)((p.N + BN - 1) / BN);
    const size_t lds = (size_t)STAGES * (BM + BN) * BK;
    auto k = qgemm_kernel<MODE, BM, BN, BK, WGM, WGN, STAGES, 1, false, DT_BF16, true>;
    static std::atomic<uint64_t> attr_set{0};
    if (!device_flag_test(attr_set)) {
        hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return (int)e;
        device_flag_set(attr_set);
    }
    hipLaunchKernelGGL(k, dim3((unsigned)(tiles_m * tiles_n), 1, (unsigned)p.splits), dim3(WGM * WGN * 64), lds, st, p, tiles_m, tiles_n);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return (int)e;
    constexpr int DT = MODE == MODE_BF16 ? DT_BF16 : DT_F16;
    splitk_launch(p.M, p.N, [&](auto w, dim3 g, dim3 b) { hipLaunchKernelGGL(gemm16_splitk_reduce_kernel<decltype(w)::value>, g, b, 0, st, p, DT); });
    return (int)hipGetLastError();
}

template <int MODE>
static int launch16(const QgemmParams& p, const Gemm16Plan& pl, hipStream_t st)
{
    if (pl.cfg >= OPSNN_VARIANT_I8_WIDE8 && pl.cfg <= OPSNN_VARIANT_I8_WIDE11) return launch_16_wide(p, pl.cfg, MODE == MODE_BF16, st);
    if (pl.splits > 1) {
        if (pl.cfg == OPSNN_VARIANT_I8_T64) return launch_split16<MODE, 64, 64, 2, 2, 5>(p, st);
        return launch_split16<MODE, 128, 128, 2, 4, 4>(p, st);
    }
    constexpr int DT = MODE == MODE_BF16 ? DT_BF16 : DT_F16;
    switch (pl.cfg) {
        case OPSNN_VARIANT_I8_T64: return qgemm_launch<MODE, 64, 64, 128, 2, 2, 5, 1>(p, 1, DT, st);
        case OPSNN_VARIANT_I8_T128: return qgemm_launch<MODE, 128, 128, 128, 2, 4, 4, 1>(p, 1, DT, st);
        case OPSNN_VARIANT_I8_T128x256: return qgemm_launch<MODE, 128, 256, 128, 2, 4, 3, 1>(p, 1, DT, st);
        case OPSNN_VARIANT_I8_T192: return qgemm_launch<MODE, 192, 256, 128, 2, 4, 2, 1>(p, 1, DT, st);
        case OPSNN_VARIANT_I8_256_W8_K128: return qgemm_launch<MODE, 256, 256, 128, 2, 4, 2, 1>(p, 1, DT, st);
        default: return qgemm_launch<MODE, 128, 128, 128, 2, 2, 2, 1>(p, 1, DT, st);
    }
}

// One launch.  Fewer 256 x 256 tiles than CUs: tile_plan (qmm_int8.hip), whose K tiles of 128 bytes take the same time here -- half as
// many products per byte at half the rate.  Otherwise the estimates, in microseconds, of the kernels for large shapes, fitted to
// 36 drawn shapes of 613 .. 3108 rows on each of them (the product alone, steady state; median error 4 %, 3 % and 5 %):
//   four-wave kernel, tiles of 256 x 32 fn: a K tile of 64 takes (0.137 + 0.057 * share of the CUs at work) fn, 5.8 a round beside
//   (4096^3: 99 us in one round of 256 x 256 tiles = 1.39 Pflop/s; 2048 x 4096 x 11008: 134 us in one round of 256 x 352);
//   eight waves on 256 x 256 tiles: 0.140 + 0.065 times 8, taken from 5 us below the others on (4 for an odd N, whose rows cost the four-wave kernel's
//   stores from the registers more): ahead of the four-wave form of that tile, 0.95 of its time, up to K = 2048, and behind it, 1.02, from there
//   to 9000.  Of 240 calls of 600 .. 4096 rows timed on all six tilings 6 take 5 % longer than on the best one, 18 where the estimates alone
//   decide (2962 x 2432 x 9176 144 us there and 132 on the four-wave kernel, 2766 x 2048 x 17360 192 and 178);
//   128 x 128 tiles, two on a CU: 1.14 a K tile.  (0.65 alone on a CU, 1.0 for two was the estimate before: 775 x 11264 x 22888 was
//   planned on them with 472 us and took 611, the eight-wave kernel takes 557.)
static Gemm16Plan one_launch(int64_t M, int64_t N, int64_t K)
{
    const int64_t cus = 256, kt = K / 64, tm = (M + 255) / 256;
    Gemm16Plan best;
    if (const TilePlan t = tile_plan(M, N, 2 * K, 1, true, false); t.variant) {
        best.cfg = t.variant; best.splits = t.splits; best.us = t.us;
        return best;
    }
    double least = 1e30;
    auto offer = [&](int cfg, double us, double doubt = 0.0) { if (us + doubt < least) { best.cfg = cfg; best.us = us; least = us + doubt; } };
    auto rounds = [&](int64_t tiles, int64_t slots, double tile, double share, double beside) {
        const int64_t full = tiles / slots, rest = tiles % slots;
        return (double)full * ((double)kt * (tile + share) + beside) + (rest ? (double)kt * (tile + share * (double)rest / (double)slots) + beside : 0.0);
    };
    for (int fn = 8; fn <= 11; fn++) offer(fn, rounds(tm * ((N + 32 * fn - 1) / (32 * fn)), cus, 0.1372 * fn, 0.0567 * fn, 5.8) + 3.7);
    offer(OPSNN_VARIANT_I8_256_W8_K128, rounds(tm * ((N + 255) / 256), cus, 1.122, 0.516, 5.6) - 6.0, N % 2 ? 4.0 : 5.0);
    offer(OPSNN_VARIANT_I8_128, rounds(((M + 127) / 128) * ((N + 127) / 128), 2 * cus, 0.108, 1.031, 0.0) + 5.0);
    return best;
}

// Two launches where one ends in a round of the chip that is nearly empty: the columns (or rows) whose tiles make whole rounds, and the
// rest on what is best for that.  Only where the estimate of one is a tenth above the time of its products in whole rounds, and where
// two are estimated below 0.95 of it.  (A whole call with its pass over the weight, int4 bf16: 775 x 11264 x 22888 739 -> 502 us, 997 x 8512 x 23552
// 543 -> 405, 1488 x 6912 x 15680 397 -> 309, 2877 x 3712 x 7424 177 -> 146; of 62 drawn calls that fill the chip nine are 1.16 to 1.28
// times as fast and none is slower by more than 3 %.)
Gemm16Plan gemm16_plan(int64_t M, int64_t N, int64_t K)
{
    Gemm16Plan best = one_launch(M, N, K);
    const int64_t cus = 256, kt = K / 64, tm = (M + 255) / 256;
    if (M <= 128 || N <= 128 || tm * ((N + 255) / 256) < cus) return best;   // (tile_plan chose)
    if (best.us < 1.1 * ((double)kt * (double)M * (double)N * (0.194 / (256.0 * 32.0 * 256.0)) + 9.5)) return best;
    const double most = 0.95 * best.us;
    Gemm16Plan two = best;
    two.us = most;
    auto consider = [&](int cfg, int64_t m, int64_t n, double us) {
        if (us >= two.us || (m == M && n == N)) return;
        const Gemm16Plan rest = one_launch(m < M ? M - m : M, n < N ? N - n : N, K);
        if (us + rest.us + 4.0 >= two.us) return;
        two.cfg = cfg; two.splits = 1; two.us = us + rest.us + 4.0;
        two.rows = m < M ? m : 0; two.cols = n < N ? n : 0;
        two.rest_cfg = rest.cfg; two.rest_splits = rest.splits;
    };
    for (int fn = 8; fn <= 11; fn++) {
        const int64_t width = 32 * fn, tn = (N + width - 1) / width, full = tm * tn / cus;
        if (full < 1) continue;
        const double us = (double)full * ((double)kt * 0.1939 * fn + 5.8) + 3.7;
        if (const int64_t c = full * cus / tm; c * width < N) consider(fn, M, c * width, us);
        if (const int64_t r = full * cus / tn; r > 0 && r * 256 < M) consider(fn, r * 256, N, us);
    }
    return two.us < most ? two : best;
}

int launch_gemm16(QgemmParams p, const Gemm16Plan& pl, bool bf16, float* part, hipStream_t st)
{
    if (p.KB % 128 != 0 || p.KB < 128) return OPSNN_NOT_TAKEN;
    if (((uintptr_t)p.a | (uintptr_t)p.b | (uint64_t)p.lda | (uint64_t)p.ldb) % 16) return OPSNN_NOT_TAKEN;
    if (256 * p.lda >= (1ll << 31) || 352 * p.ldb >= (1ll << 31)) return OPSNN_NOT_TAKEN;   // 32-bit offsets inside a tile
    p.part = (int32_t*)part;
    auto launch = [&](const QgemmParams& q, const Gemm16Plan& of) { return bf16 ? launch16<MODE_BF16>(q, of, st) : launch16<MODE_F16>(q, of, st); };
    QgemmParams q = p;
    q.splits = pl.splits;
    if (pl.rows) q.M = pl.rows;
    if (pl.cols) q.N = pl.cols;
    int rc = launch(q, pl);
    if (rc != 0 || (!pl.rows && !pl.cols)) return rc;
    Gemm16Plan rest;
    rest.cfg = pl.rest_cfg; rest.splits = q.splits = pl.rest_splits;
    q.M = p.M - pl.rows; q.N = p.N - pl.cols;
    q.a = p.a + pl.rows * p.lda;
    q.b = p.b + pl.cols * p.ldb;
    q.out = (uint16_t*)p.out + pl.rows * p.ldc + pl.cols;
    if (p.bias) q.bias = (const char*)p.bias + pl.cols * (p.bias_dt == DT_F32 ? 4 : 2);
    return launch(q, rest);
}

}  // namespace opsnn
