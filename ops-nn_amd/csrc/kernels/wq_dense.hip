// Weight-only matmul with many rows of x: the weight is dequantised ONCE per call to x's own type, K-contiguous, into the
// workspace, and the product is a dense 16-bit one (gemm16.hip).
//
//   w16[n][k] = T(T(w[k,n] + offset[g,n]) * scale[g,n])      the two roundings of the formula, as in wqmm_stream.hip.h
//
// Cost of the pass: half or one byte read and two bytes written per weight; the streaming kernels dequantise in registers
// once per 256 rows instead, so the pass pays from a few hundred rows on, and from far fewer where those kernels do not
// run (N no multiple of 32, K no whole number of x slabs, groups of 64, [K, N] storage): it takes every layout, group and N.
#include "gemm16.h"
#include "launch.h"
#include "wq_kn.hip.h"
#include "wqmm_stream.hip.h"

extern "C" int opsnn_wq_tile_min();   // dispatch.hip
namespace opsnn {

// [N, K] storage: a lane turns 8 consecutive k of one row into 16 bytes; a wave covers 512 k of a row per step.
template <int XDT, int WBITS, bool HAS_OFF>
__global__ __launch_bounds__(256) void wq_dequant_nk_kernel(WqParams p, uint16_t* __restrict__ out, int steps)
{
    const int lane = threadIdx.x & 63;
    const int64_t n = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);   // (N on grid.x: grid.y ends at 65535)
    if (n >= p.N) return;
    const uint8_t* w = p.w + n * p.ldw;
    const uint16_t* sc = p.scale + n * p.s_cs;
    const uint16_t* of = HAS_OFF ? p.offset + n * p.s_cs : nullptr;
    const DqConst dqc = make_dq_const();
    const int Ki = (int)p.K, groupi = (int)p.group;
#pragma unroll 4
    for (int s = 0; s < steps; s++) {
        const int k = ((int)blockIdx.y * steps + s) * 512 + lane * 8;
        if (k >= Ki) break;
        v4i q = {0, 0, 0, 0};
        if constexpr (WBITS == 4) q[0] = *(const int*)(w + k / 2);
        else { const v2i t = *(const v2i*)(w + k); q[0] = t[0]; q[1] = t[1]; }
        const int g = p.group_shift >= 0 ? k >> p.group_shift : k / groupi;
        const uint16_t sb = sc[(int64_t)g * p.s_rs], ob = HAS_OFF ? of[(int64_t)g * p.s_rs] : (uint16_t)0;
        *(v4i*)(out + n * p.K + k) = dequant8<XDT, WBITS, HAS_OFF, true>(q, 0, sb, ob, dqc);
    }
}

// [K, N] storage: a lane takes 8 rows of k and 8 neighbouring columns (dequant_8x8) and writes, per column, 16 bytes of 8
// consecutive k; 16 lanes side by side in k make 256 contiguous bytes of an output row.
template <int XDT, int WBITS, bool HAS_OFF>
__global__ __launch_bounds__(256) void wq_dequant_kn_kernel(WqParams p, uint16_t* __restrict__ out)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t k0 = (int64_t)blockIdx.y * 128 + (lane & 15) * 8;
    const int64_t n0 = ((int64_t)blockIdx.x * 16 + wave * 4 + (lane >> 4)) * 8;
    if (k0 >= p.K || n0 >= p.N) return;
    const int cols = p.N - n0 < 8 ? (int)(p.N - n0) : 8;
    const int g = p.group_shift >= 0 ? (int)k0 >> p.group_shift : (int)k0 / (int)p.group;
    // codes: row i of the block in q[i] (int4: one dword, int8: two)
    constexpr int DW = WBITS / 4;
    uint32_t q[8][DW];
    const uint8_t* src = p.w + k0 * p.ldw + n0 * WBITS / 8;
    if (cols == 8) {
#pragma unroll
        for (int i = 0; i < 8; i++) __builtin_memcpy(q[i], src + i * p.ldw, 4 * DW);
    } else {   // the matrix edge: byte by byte (4-bit: N is even)
        for (int i = 0; i < 8; i++) {
            uint8_t b[4 * DW] = {};
            for (int j = 0; j * 8 / WBITS < cols; j++) b[j] = src[i * p.ldw + j];
            __builtin_memcpy(q[i], b, 4 * DW);
        }
    }
    uint16_t sb[8], ob[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const int64_t n = n0 + (j < cols ? j : cols - 1);
        sb[j] = p.scale[(int64_t)g * p.s_rs + n * p.s_cs];
        ob[j] = HAS_OFF ? p.offset[(int64_t)g * p.s_rs + n * p.s_cs] : (uint16_t)0;
    }
    uint32_t o[8][4], scw[4], ofw[4];   // o[column][pair of k]
#pragma unroll
    for (int t = 0; t < 4; t++) {
        scw[t] = sb[2 * t] | ((uint32_t)sb[2 * t + 1] << 16);
        ofw[t] = ob[2 * t] | ((uint32_t)ob[2 * t + 1] << 16);
    }
    dequant_8x8<XDT, WBITS, HAS_OFF>(q, scw, ofw, o);
#pragma unroll
    for (int j = 0; j < 8; j++)
        if (j < cols) *(v4i*)(out + (n0 + j) * p.K + k0) = (v4i){(int)o[j][0], (int)o[j][1], (int)o[j][2], (int)o[j][3]};
}

template <int XDT, int WBITS, bool HAS_OFF>
static int launch_dequant(const WqParams& p, bool kn, uint16_t* out, hipStream_t st)
{
    if (kn) {
        const dim3 grid((unsigned)((p.N + 127) / 128), (unsigned)((p.K + 127) / 128));
        hipLaunchKernelGGL((wq_dequant_kn_kernel<XDT, WBITS, HAS_OFF>), grid, dim3(256), 0, st, p, out);
    } else {
        const int steps = 4;
        const dim3 grid((unsigned)((p.N + 3) / 4), (unsigned)((p.K + 512 * steps - 1) / (512 * steps)));
        hipLaunchKernelGGL((wq_dequant_nk_kernel<XDT, WBITS, HAS_OFF>), grid, dim3(256), 0, st, p, out, steps);
    }
    return (int)hipGetLastError();
}

static uint64_t dense_weight_bytes(const OpsnnWqmmArgs& a) { return ((uint64_t)a.N * (uint64_t)a.K * 2 + 255) / 256 * 256; }

// What the many-rows streaming kernel takes, in us: a workgroup of 128 columns and R rows (64, 128, 192 or 256) walks 4096 k in
// 14 + 0.21 R (measured 27, 38, 52 and 67; a quarter less where few CUs have one), a CU at a time; rows as wq_narrow_slab_rows deals them, or in passes of 256.  With
// more than 128 rows and a K that is no whole number of x rounds of those instances, three times that.
static double rows_kernel_us(const OpsnnWqmmArgs& a, int wbits, int64_t group)
{
    const int64_t wgs = (a.N + 127) / 128, kx = 2 * 4 * (128 / wbits), slab = wq_narrow_slab_rows(a.M, a.N, true);
    const int64_t ks = wq_rows_ksplit(wbits, a.M, a.N, a.K, group, true);
    auto launch_us = [&](int64_t rows, int64_t slabs) {
        const int64_t r = (rows + 63) / 64 * 64, n = wgs * slabs * ks;
        const double rounds = n < 256 ? 0.75 + 0.25 * (double)n / 256.0 : (double)((n + 255) / 256);
        return rounds * (double)a.K / (4096.0 * (double)ks) * (14.0 + 0.21 * (double)r) * (r > 128 && a.K % (4 * kx) != 0 ? 3.0 : 1.0);
    };
    const double part_us = ks > 1 ? 4.0 + 8.0 * (double)ks * (double)a.M * (double)a.N / 5.0e6 : 0.0;
    if (slab) return launch_us(slab, (a.M + slab - 1) / slab) + part_us;
    return (double)(a.M / 256) * launch_us(256, 1) + (a.M % 256 ? launch_us(a.M % 256, 1) : 0.0) + part_us;
}

// Does the call run on this route?  Looks at what phase 1 knows (shapes, types, layouts, addresses), so that both phases agree.
//
// The pass moves 2.5 (8-bit weights: 3) bytes per weight at 5 TB/s, the product takes what gemm16_plan estimates.  Against
// it stands the many-rows streaming kernel where it runs (wqmm.hip: [N, K] storage, N % 32 == 0, whole x slabs and groups of
// whole chunks); everywhere else the general kernel re-reads the weight per 64 rows at a fraction of its speed, and this
// route takes every call of more than 64 rows.  (Measured: 1999 x 4096 x 11008 bf16 x int4 228 -> 156 us, [K, N] storage
// 613 -> 162; 700 x 4096 x 11008 134 -> 106; 1024 x 8192 x 28672 497 against 499, 512 rows 254 against 330.)
bool wq_dense_wanted(const OpsnnWqmmArgs& a)
{
    if (a.w_dtype != DT_I4 && a.w_dtype != DT_I8) return false;
    if (a.x_dtype != DT_F16 && a.x_dtype != DT_BF16) return false;
    if (a.scale_dtype != a.x_dtype || a.force_variant == OPSNN_VARIANT_PLAIN) return false;
    if (opsnn_wq_tile_min() <= 128) return false;   // (test hook: such calls are sent to the tile kernel of wqmm_tile.hip)
    if (a.M <= 64 || a.K % 64 != 0 || a.N < 128 || (uintptr_t)a.x % 16) return false;
    if (a.K >= (1ll << 22) || a.N >= (1ll << 24)) return false;   // (grids: K / 128 on grid.y, 64 threads per column on grid.x)
    if (a.group > 0 && a.group % 8 != 0) return false;
    const bool nk = a.w.row_stride == 1 && a.w.col_stride == a.K, kn = a.w.col_stride == 1 && a.w.row_stride == a.N;
    if (!nk && !kn) return false;
    if (a.w_dtype == DT_I4 && !nk && a.N % 2 != 0) return false;
    const int wbits = a.w_dtype == DT_I4 ? 4 : 8;
    const int64_t kc = 4 * (128 / wbits);
    const int64_t cpg = a.group > 0 && a.group < a.K ? a.group / kc : 1;
    const bool rows_kernel = nk && a.N % 32 == 0 && a.N >= 256 && a.K % (2 * kc) == 0 &&
                             (a.group <= 0 || a.group >= a.K || (a.group % kc == 0 && (cpg & (cpg - 1)) == 0));
    if (!rows_kernel) return true;
    const double rows_us = rows_kernel_us(a, wbits, a.group > 0 && a.group < a.K ? a.group : a.K);
    const double dense_us = 2.0 + (double)a.N * (double)a.K * (2.0 + wbits / 8.0) / 5.0e6 + gemm16_plan(a.M, a.N, a.K, 1).us;
    return dense_us < rows_us;
}
uint64_t wq_dense_workspace(const OpsnnWqmmArgs& a)
{
    const Gemm16Plan pl = gemm16_plan(a.M, a.N, a.K, 1);
    return dense_weight_bytes(a) + gemm16_part_bytes(pl, a.M, a.N, 1);
}

bool weight_cache_on();   // weight_cache.hip
const void* weight_cache_get(const void* src, int64_t K, int64_t N, int bits, int64_t nb, hipStream_t st);
int launch_wqmm_mfma(const OpsnnWqmmArgs& a, hipStream_t st);   // wqmm.hip

int launch_wq_dense(const OpsnnWqmmArgs& a, hipStream_t st)
{
    if (!a.workspace || !wq_dense_wanted(a)) return OPSNN_NOT_TAKEN;
    const int wbits = a.w_dtype == DT_I4 ? 4 : 8;
    const bool kn = a.w.row_stride != 1;
    if (kn && weight_cache_on()) {
        // a caller who keeps K-contiguous copies in the weight cache: where that form runs on the streaming kernel, so does the
        // copy (128 x 8192 x 28672 int4: 75 us, 329 with the pass here); phase 1 has left room for its partial sums
        OpsnnWqmmArgs b = a;
        b.w.row_stride = 1; b.w.col_stride = a.K;
        if (!wq_dense_wanted(b) && (b.w.ptr = weight_cache_get(a.w.ptr, a.K, a.N, wbits, 1, st)) != nullptr) {
            const int rc = launch_wqmm_mfma(b, st);
            if (rc != OPSNN_NOT_TAKEN) return rc;
        }
    }
    uint16_t* w16 = (uint16_t*)a.workspace;
    WqParams p{};
    p.w = (const uint8_t*)a.w.ptr;
    p.ldw = (kn ? a.w.row_stride : a.w.col_stride) * wbits / 8;
    p.scale = (const uint16_t*)a.scale.ptr; p.offset = (const uint16_t*)a.offset;
    p.s_rs = a.scale.row_stride; p.s_cs = a.scale_n == 1 ? 0 : a.scale.col_stride;
    p.M = a.M; p.N = a.N; p.K = a.K;
    p.group = a.group > 0 ? a.group : a.K;
    p.group_shift = (p.group & (p.group - 1)) == 0 ? __builtin_ctzll((unsigned long long)p.group) : p.group >= p.K ? 31 : -1;
    const bool f16 = a.x_dtype == DT_F16;
    int rc;
    if (f16) {
        if (wbits == 4) rc = a.offset ? launch_dequant<DT_F16, 4, true>(p, kn, w16, st) : launch_dequant<DT_F16, 4, false>(p, kn, w16, st);
        else rc = a.offset ? launch_dequant<DT_F16, 8, true>(p, kn, w16, st) : launch_dequant<DT_F16, 8, false>(p, kn, w16, st);
    } else {
        if (wbits == 4) rc = a.offset ? launch_dequant<DT_BF16, 4, true>(p, kn, w16, st) : launch_dequant<DT_BF16, 4, false>(p, kn, w16, st);
        else rc = a.offset ? launch_dequant<DT_BF16, 8, true>(p, kn, w16, st) : launch_dequant<DT_BF16, 8, false>(p, kn, w16, st);
    }
    if (rc != 0) return rc;
    const Gemm16Plan pl = gemm16_plan(a.M, a.N, a.K, 1);
    QgemmParams g{};
    g.a = (const int8_t*)a.x; g.b = (const int8_t*)w16;
    g.lda = 2 * a.K; g.ldb = 2 * a.K; g.KB = 2 * a.K;
    g.out = a.y; g.M = a.M; g.N = a.N; g.ldc = a.N;
    g.bias = a.bias; g.bias_dt = a.bias_dtype;
    return launch_gemm16(g, pl, !f16, 1, a.x_dtype, (float*)((char*)a.workspace + dense_weight_bytes(a)), st);
}

}  // namespace opsnn
