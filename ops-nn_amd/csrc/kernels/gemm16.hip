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

// Fewer 256 x 256 tiles than CUs: tile_plan (qmm_int8.hip), whose K tiles of 128 bytes take the same time here -- half as many
// products per byte at half the rate.  Otherwise the estimate, in microseconds, of the two kernels for large shapes, fitted to
// random operands, K = 4096 .. 18432 (profiles/tile_plans.txt: the pass and this product together, 41 calls of 100 .. 1999 rows, 37 within
// 3 % of the fastest tile, the worst 8 % behind):
//   four-wave kernel: 0.185 us per 32 columns of tile width and 64-element K tile, 8 us a round beside (4096^3: 99 us in one
//   round of 256 x 256 tiles = 1.39 Pflop/s; 2048 x 4096 x 11008: 134 us in one round of 256 x 352);
//   128 x 128 tiles: 0.65 us per K tile alone on a CU, 1.0 us for two that share one, 6 us beside.
Gemm16Plan gemm16_plan(int64_t M, int64_t N, int64_t K)
{
    const int64_t cus = 256, kt = K / 64;
    Gemm16Plan best;
    if (const TilePlan t = tile_plan(M, N, 2 * K, 1, true, false); t.variant) {
        best.cfg = t.variant; best.splits = t.splits; best.us = t.us;
        return best;
    }
    best.us = 1e30;
    const int64_t tm = (M + 255) / 256;
    for (int fn = 8; fn <= 11; fn++) {
        const int64_t tiles = tm * ((N + 32 * fn - 1) / (32 * fn));
        const double us = (double)((tiles + cus - 1) / cus) * (0.185 * fn * (double)kt + 8.0);
        if (us < best.us) { best.cfg = fn; best.us = us; }
    }
    const int64_t t128 = ((M + 127) / 128) * ((N + 127) / 128), per_cu = (t128 + cus - 1) / cus;
    const double us = (double)kt * ((double)(per_cu / 2) * 1.0 + (double)(per_cu % 2) * 0.65) + 6.0;
    if (us < best.us) { best.cfg = OPSNN_VARIANT_I8_128; best.us = us; }
    return best;
}

int launch_gemm16(QgemmParams p, const Gemm16Plan& pl, bool bf16, float* part, hipStream_t st)
{
    if (p.KB % 128 != 0 || p.KB < 128) return OPSNN_NOT_TAKEN;
    if (((uintptr_t)p.a | (uintptr_t)p.b | (uint64_t)p.lda | (uint64_t)p.ldb) % 16) return OPSNN_NOT_TAKEN;
    if (256 * p.lda >= (1ll << 31) || 352 * p.ldb >= (1ll << 31)) return OPSNN_NOT_TAKEN;   // 32-bit offsets inside a tile
    p.splits = pl.splits;
    p.part = (int32_t*)part;
    return bf16 ? launch16<MODE_BF16>(p, pl, st) : launch16<MODE_F16>(p, pl, st);
}

}  // namespace opsnn
