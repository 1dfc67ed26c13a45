// MXFP4 (fp4 e2m1 x fp4 e2m1, one e8m0 scale per 32 elements of K) with few rows of x1: the decode shape, a stream over x2.
//
//   out[m,n] = cast( sum_k (x1[m,k] * 2^(s1[m,k/32]-127)) * (x2[k,n] * 2^(s2[k/32,n]-127)) + bias[n] )
//
// Formula: matmul/quant_batch_matmul_v3/tests/assets/qbmmv3_kernel_golden.py:153-234.
//
// The tile kernel owns 128 rows of x1 and 128 columns per workgroup: with one to a few dozen rows it leaves most CUs without a
// workgroup and each of the others with one serial chain of copies.  Here a wave streams x2 straight into registers: lane
// (r = lane % 16, q = lane / 16) holds 16 bytes, one scale block, of column 16 j + r; four lanes cover the 128 elements of one
// v_mfma_scale_f32_16x16x128_f8f6f4, which takes the operands and both scale bytes as they lie in memory.  x1's pieces come the
// same way (from L2: every workgroup reads the few rows of x1 once), so the loop has no LDS, no barrier and no conversion.
//
// Work split: a workgroup owns 16 NB columns and 16 MB rows; its NW waves take units of S steps of 128 elements in turn, two units
// in flight, and meet in LDS at the end, added in wave order.  K is cut by waves only, so a call is one launch.
// K need be no multiple of 128: what is left behind the last whole unit goes to the waves step by step, requested ahead of the
// loop, lanes past the end of K with zeros for x1 and a unit scale on both sides.
#include <cmath>

#include "launch.h"
#include "common.hip.h"

namespace opsnn {
namespace {

struct Mx4RowsParams {
    const uint8_t *a, *b;               // x1 [M, K / 2] and x2 as [N, K / 2] bytes
    int64_t lda, ldb, a_bs, b_bs;       // bytes
    const uint8_t *sa, *sb;             // e8m0 [M, K / 32], [N, K / 32]
    int64_t sa_rs, sb_rs, sa_bs, sb_bs;
    void* out; int out_dt;
    int M, N, blocks;                   // blocks of 32 along K
    const float* bias; int64_t bias_bs;
};

template <int MB, int NB, int NW, int S>
__global__ __launch_bounds__(NW * 64) void mxfp4_rows_kernel(Mx4RowsParams p)
{
    extern __shared__ __attribute__((aligned(16))) float red[];   // [NW][NB * MB][256]
    typedef uint32_t words_t __attribute__((ext_vector_type(S == 1 ? 2 : S)));   // a row's scale bytes of a unit
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, q = lane >> 4;
    const int n0 = (int)blockIdx.x * (16 * NB), m0 = (int)blockIdx.y * (16 * MB);
    const int64_t bz = blockIdx.z;
    const uint8_t* A = p.a + bz * p.a_bs;
    const uint8_t* B = p.b + bz * p.b_bs;
    const uint8_t* SA = p.sa + bz * p.sa_bs;
    const uint8_t* SB = p.sb + bz * p.sb_bs;
    // byte offsets of this lane's rows (rows and columns past the edge repeat the last one; the launcher keeps them below 2^32)
    uint32_t wo[NB], wso[NB], xo[MB], xso[MB];
#pragma unroll
    for (int j = 0; j < NB; j++) {
        const int n = n0 + 16 * j + r < p.N ? n0 + 16 * j + r : p.N - 1;
        wo[j] = (uint32_t)(n * p.ldb);
        wso[j] = (uint32_t)(n * p.sb_rs);
    }
#pragma unroll
    for (int b = 0; b < MB; b++) {
        const int m = m0 + 16 * b + r < p.M ? m0 + 16 * b + r : p.M - 1;
        xo[b] = (uint32_t)(m * p.lda);
        xso[b] = (uint32_t)(m * p.sa_rs);
    }
    v4f acc[NB][MB];
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
        for (int b = 0; b < MB; b++) acc[j][b] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
    auto mma = [&](const v4i (&w)[NB], const v4i (&x)[MB], const uint32_t (&ws)[NB], const uint32_t (&xs)[MB]) {   // scale bytes in bits 0..7
#pragma unroll
        for (int j = 0; j < NB; j++)
#pragma unroll
            for (int b = 0; b < MB; b++) {
                const v8i wf = {w[j][0], w[j][1], w[j][2], w[j][3], 0, 0, 0, 0}, xf = {x[b][0], x[b][1], x[b][2], x[b][3], 0, 0, 0, 0};
                acc[j][b] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf, xf, acc[j][b], 4, 4, 0, (int)ws[j], 0, (int)xs[b]);
            }
    };

    // behind the last whole unit: step `tail` of what is left, for this wave or (not live) nobody
    const int units = p.blocks / (4 * S), rest = p.blocks - units * 4 * S, tails = (rest + 3) / 4;
    const int tail = (wave + NW - units % NW) % NW;
    const bool has_tail = tail < tails;
    v4i tw[NB], tx[MB];
    uint32_t tws[NB], txs[MB];
    const int tblk = units * 4 * S + 4 * (has_tail ? tail : 0) + q;
    const bool inside = tblk < p.blocks;
    if (has_tail) {
        const uint32_t at = (uint32_t)(inside ? tblk : p.blocks - 1);
#pragma unroll
        for (int j = 0; j < NB; j++) { tw[j] = *(const v4i*)(B + (wo[j] + 16 * at)); tws[j] = SB[wso[j] + at]; }
#pragma unroll
        for (int b = 0; b < MB; b++) { tx[b] = *(const v4i*)(A + (xo[b] + 16 * at)); txs[b] = SA[xso[b] + at]; }
    }

    if (wave < units) {
        v4i w[2][S][NB], x[2][S][MB];
        words_t ws[2][NB], xs[2][MB];
        auto fetch = [&](auto jc, int u) {
            constexpr int i = decltype(jc)::value;
            const uint32_t u1 = (uint32_t)(u < units ? u : units - 1), k = u1 * (64 * S) + 16 * q, ks = u1 * (4 * S);   // past the end: a harmless reload
#pragma unroll
            for (int j = 0; j < NB; j++) __builtin_memcpy(&ws[i][j], SB + (wso[j] + ks), 4 * S);
#pragma unroll
            for (int b = 0; b < MB; b++) __builtin_memcpy(&xs[i][b], SA + (xso[b] + ks), 4 * S);
#pragma unroll
            for (int s = 0; s < S; s++) {
#pragma unroll
                for (int j = 0; j < NB; j++) w[i][s][j] = *(const v4i*)(B + (wo[j] + k + 64 * s));
#pragma unroll
                for (int b = 0; b < MB; b++) x[i][s][b] = *(const v4i*)(A + (xo[b] + k + 64 * s));
            }
        };
        auto unit = [&](auto jc) {
            constexpr int i = decltype(jc)::value;
#pragma unroll
            for (int s = 0; s < S; s++) {
                uint32_t a[NB], c[MB];
#pragma unroll
                for (int j = 0; j < NB; j++) a[j] = ws[i][j][s] >> (8 * q);
#pragma unroll
                for (int b = 0; b < MB; b++) c[b] = xs[i][b][s] >> (8 * q);
                mma(w[i][s], x[i][s], a, c);
            }
        };
        using I0 = std::integral_constant<int, 0>;
        using I1 = std::integral_constant<int, 1>;
        fetch(I0{}, wave);
        fetch(I1{}, wave + NW);
        for (int u = wave; u < units; u += 2 * NW) {
            unit(I0{});
            fetch(I0{}, u + 2 * NW);
            if (u + NW >= units) break;
            unit(I1{});
            fetch(I1{}, u + 3 * NW);
        }
    }
    if (has_tail) {
        if (!inside) {
#pragma unroll
            for (int j = 0; j < NB; j++) tws[j] = 127;
#pragma unroll
            for (int b = 0; b < MB; b++) { tx[b] = (v4i){0, 0, 0, 0}; txs[b] = 127; }
        }
        mma(tw, tx, tws, txs);
    }

    // acc[j][b][e]: n = n0 + 16 j + 4 q + e, m = m0 + 16 b + r, over this wave's part of K
    float* mine = red + wave * (NB * MB * 256) + lane * 4;
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
        for (int b = 0; b < MB; b++) *(v4f*)(mine + (j * MB + b) * 256) = acc[j][b];
    __syncthreads();
    for (int t = tid; t < NB * MB * 64; t += NW * 64) {
        const float* all = red + t * 4;
        v4f sum = *(const v4f*)all;
#pragma unroll
        for (int i = 1; i < NW; i++) {
            const v4f o = *(const v4f*)(all + i * (NB * MB * 256));
#pragma unroll
            for (int e = 0; e < 4; e++) sum[e] = sum[e] + o[e];
        }
        const int j = (t >> 6) / MB, b = (t >> 6) % MB;
        const int m = m0 + 16 * b + (t & 15), n = n0 + 16 * j + 4 * ((t >> 4) & 3);
        if (m >= p.M || n >= p.N) continue;
        if (p.bias) {
#pragma unroll
            for (int e = 0; e < 4; e++) sum[e] = sum[e] + p.bias[bz * p.bias_bs + (n + e < p.N ? n + e : p.N - 1)];
        }
        const int64_t at = (bz * p.M + m) * p.N + n;
        if (p.out_dt == DT_F32) {
            float* dst = (float*)p.out + at;
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (n + e < p.N) dst[e] = sum[e];
        } else {
            const v4us o = p.out_dt == DT_BF16 ? pack4_b16<DT_BF16>(sum) : pack4_b16<DT_F16>(sum);
            uint16_t* dst = (uint16_t*)p.out + at;
            if (n + 3 < p.N) __builtin_memcpy(dst, &o, 8);
            else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (n + e < p.N) dst[e] = o[e];
            }
        }
    }
}

constexpr int64_t MX4_MAX_ROWS = 128;

template <int MB, int NB, int NW, int S>
int launch_one(const Mx4RowsParams& p, int64_t batch, hipStream_t st)
{
    const dim3 grid((unsigned)((p.N + 16 * NB - 1) / (16 * NB)), (unsigned)((p.M + 16 * MB - 1) / (16 * MB)), (unsigned)batch);
    constexpr size_t lds = (size_t)NW * NB * MB * 1024;
    auto k = mxfp4_rows_kernel<MB, NB, NW, S>;
    if constexpr (lds > 65536) {
        static std::atomic<uint64_t> attr_set{0};   // one bit per device: the attribute belongs to the (kernel, device) pair
        if (!device_flag_test(attr_set)) {
            hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            if (e != hipSuccess) return (int)e;
            device_flag_set(attr_set);
        }
    }
    note_route("mxfp4_rows");
    hipLaunchKernelGGL(k, grid, dim3(NW * 64), lds, st, p);
    return (int)hipGetLastError();
}

}  // namespace

// Does a call run here (both phases ask; operands K-contiguous, or re-laid out so by then)?
//
// Up to 16 rows always: 1 x 7040 x 10176 32.5 us on the tile kernel and 10.7 here, 16 x 8192 x 8192 17.2 and 11.7, 16 x 4096 x 28672
// 19.5 and 19.4, 16 x 1984 x 1056 in 8 batches (K padded by four launches there) 21.6 and 6.8.  With more rows each workgroup reads x1
// as often as its columns' share of x2, and a large x2 is faster on the tiles where those can cut K: the estimate below, fitted to 210
// calls of 17 .. 128 rows, each as the geometric mean of its time with the weight from memory and from the last-level cache (median
// error 7 %), against that of mxfp4_tile_plan (24 x 4480 x 15680 24.1 there and 14.4 here, 64 x 4480 x 1280 17.7 and 7.7, but
// 64 x 4096 x 28672 22.0 and 43.8, 50 x 18176 x 1088 13.0 and 25.3).
bool mxfp4_rows_wanted(const OpsnnQmmArgs& a)
{
    if (a.x1_dtype != DT_E2M1 || a.x2_dtype != DT_E2M1 || a.force_variant != 0) return false;
    if (a.M > MX4_MAX_ROWS || a.N < 256 || a.K < 128 || a.K % 32 != 0 || a.K > (1 << 30) || a.N > (1 << 30) || a.batch > 65535) return false;
    // (32-bit lane offsets)
    if (a.x1.row_stride < 0 || a.x2.col_stride < 0 || a.x1_scale_mat.row_stride < 0 || a.x2_scale_mat.row_stride < 0) return false;
    if (a.x1.row_stride / 2 >= (1ll << 32) / MX4_MAX_ROWS || a.N * ((a.x2.row_stride == 1 ? a.x2.col_stride : a.K) / 2) >= (1ll << 32)) return false;
    if (a.M <= 16) return true;
    // K steps of 128 elements in turns of eight waves; workgroups of 16 or 32 columns and up to 64 rows, two to a CU up to 32 rows
    const int64_t w1 = (a.N + 15) / 16 * a.batch, slabs = (a.M + 63) / 64, mb = a.M > 64 ? 4 : (a.M + 15) / 16;
    const int64_t nb = w1 <= 128 ? 1 : 2, wgs = (nb == 1 ? w1 : (a.N + 31) / 32 * a.batch) * slabs;
    double turns = (double)((wgs + 255) / 256);
    if (a.M <= 32 && wgs > 256) turns = wgs <= 512 ? 1.42 : 0.71 * ((double)wgs / 512.0 + (double)((wgs + 511) / 512));
    const double steps = (double)((a.K + 1023) / 1024);
    const double here = 2.05 + turns * steps * (0.276 + 0.026 * (double)(mb * nb) + 0.193 * (double)mb) +
                        (double)a.batch * (double)a.N * (double)a.K * 0.5e-6 / 5.23 * std::sqrt((double)slabs);
    return 0.98 * here < mxfp4_tile_plan(a.M, a.N, a.K, a.batch, true).us;
}
int launch_mxfp4_rows(const OpsnnQmmArgs& a, hipStream_t st)
{
    if (!mxfp4_rows_wanted(a) || a.x1.col_stride != 1 || a.x2.row_stride != 1) return OPSNN_NOT_TAKEN;
    if (a.out_dtype != DT_BF16 && a.out_dtype != DT_F16 && a.out_dtype != DT_F32) return OPSNN_NOT_TAKEN;
    if (a.bias && a.bias_dtype != DT_F32) return OPSNN_NOT_TAKEN;
    if (a.x1_scale_mat.col_stride != 2 || a.x2_scale_mat.col_stride != 2) return OPSNN_NOT_TAKEN;   // [rows, K / 64, 2]: a row's bytes contiguous
    if ((a.x1.row_stride | a.x2.col_stride | a.x1.batch_stride | a.x2.batch_stride) % 2) return OPSNN_NOT_TAKEN;
    Mx4RowsParams p{};
    p.a = (const uint8_t*)a.x1.ptr; p.b = (const uint8_t*)a.x2.ptr;
    p.lda = a.x1.row_stride / 2; p.ldb = a.x2.col_stride / 2; p.a_bs = a.x1.batch_stride / 2; p.b_bs = a.x2.batch_stride / 2;
    p.sa = (const uint8_t*)a.x1_scale_mat.ptr; p.sb = (const uint8_t*)a.x2_scale_mat.ptr;
    p.sa_rs = a.x1_scale_mat.row_stride; p.sb_rs = a.x2_scale_mat.row_stride;
    p.sa_bs = a.x1_scale_mat.batch_stride; p.sb_bs = a.x2_scale_mat.batch_stride;
    if (((uintptr_t)p.a | (uintptr_t)p.b | (uint64_t)p.lda | (uint64_t)p.ldb | (uint64_t)p.a_bs | (uint64_t)p.b_bs) % 16) return OPSNN_NOT_TAKEN;
    p.out = a.out; p.out_dt = a.out_dtype;
    p.M = (int)a.M; p.N = (int)a.N; p.blocks = (int)(a.K / 32);
    p.bias = (const float*)a.bias; p.bias_bs = a.bias_batch_stride;
    // Few columns: sixteen (eight) waves share K, so that few workgroups still have a short chain each.  Else 32 columns per
    // workgroup, or 16 where that spreads the workgroups over the 256 CUs clearly better (1 x 7040 x 10176: 318 workgroups 12.9 us,
    // 636 10.8; 1 x 8192 x 8192: 256 workgroups 10.9, 512 12.0).
    const int64_t w1 = (a.N + 15) / 16 * a.batch, w2 = (a.N + 31) / 32 * a.batch;
    const double e1 = (double)w1 / (double)((w1 + 255) / 256), e2 = (double)w2 / (double)((w2 + 255) / 256);
    if (a.M <= 16) {
        if (w1 <= 256) return launch_one<1, 1, 16, 2>(p, a.batch, st);
        return e1 > 1.1 * e2 ? launch_one<1, 1, 4, 4>(p, a.batch, st) : launch_one<1, 2, 4, 4>(p, a.batch, st);
    }
    const bool narrow = w1 <= 128;
    if (a.M <= 32) return narrow ? launch_one<2, 1, 8, 2>(p, a.batch, st) : launch_one<2, 2, 8, 2>(p, a.batch, st);
    if (a.M <= 48) return narrow ? launch_one<3, 1, 8, 2>(p, a.batch, st) : launch_one<3, 2, 8, 2>(p, a.batch, st);
    return narrow ? launch_one<4, 1, 8, 2>(p, a.batch, st) : launch_one<4, 2, 8, 2>(p, a.batch, st);
}

}  // namespace opsnn
