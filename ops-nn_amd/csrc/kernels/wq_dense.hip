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
#include "wq_cost.h"
#include "wq_kn.hip.h"
#include "wqmm_stream.hip.h"

extern "C" int opsnn_wq_tile_min();   // dispatch.hip
namespace opsnn {

// [N, K] storage: a lane turns 8 consecutive k of one row into 16 bytes; a wave covers 512 k of a row per step.
template <int XDT, int WBITS, bool HAS_OFF>
__global__ __launch_bounds__(256) void wq_dequant_nk_kernel(WqParams p, uint16_t* __restrict__ out, int steps)
{
    const int lane = threadIdx.x & 63;
    const int kblocks = ((int)p.K + 512 * steps - 1) / (512 * steps);   // (one grid dimension, K first: grid.y ends at 65535)
    const int64_t n = (int64_t)(blockIdx.x / (unsigned)kblocks) * 4 + (threadIdx.x >> 6);
    const int kb = (int)(blockIdx.x % (unsigned)kblocks);
    if (n >= p.N) return;
    const uint8_t* w = p.w + n * p.ldw;
    const uint16_t* sc = p.scale + n * p.s_cs;
    const uint16_t* of = HAS_OFF ? p.offset + n * p.s_cs : nullptr;
    const DqConst dqc = make_dq_const();
    const int Ki = (int)p.K, groupi = (int)p.group;
#pragma unroll 4
    for (int s = 0; s < steps; s++) {
        const int k = (kb * steps + s) * 512 + lane * 8;
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
        const dim3 grid((unsigned)((p.N + 3) / 4 * ((p.K + 512 * steps - 1) / (512 * steps))));
        hipLaunchKernelGGL((wq_dequant_nk_kernel<XDT, WBITS, HAS_OFF>), grid, dim3(256), 0, st, p, out, steps);
    }
    return (int)hipGetLastError();
}

// The columns go in strips whose dequantised weight takes at most 1 GiB of workspace (a vocabulary of 152064 against 8192: 2.5 GB in
// one piece).  Of the widths between half of that and all of it the one whose products have the smallest estimate: a strip that ends
// in a nearly empty round of the chip loses a tenth (1000 x 8192 x 152064: 2335 us so,
// 2315 in one piece, 2588 in five equal strips).
constexpr int64_t STRIP_BYTES = 1ll << 30;
struct DensePlan {
    int64_t strip, strips;      // columns of a strip but the last one
    Gemm16Plan full, last;
    double us;                  // the products' estimate
    uint64_t weight_bytes, part_bytes;
};
static DensePlan dense_plan(int64_t M, int64_t N, int64_t K)
{
    DensePlan best;
    best.us = 1e30;
    const int64_t most = STRIP_BYTES / (2 * K) / 256 * 256;
    for (int i = 0; i < 8; i++) {
        DensePlan d;
        d.strip = most >= N ? N : most - most * i / 16 / 256 * 256;
        if (d.strip < 256 && d.strip < N) d.strip = 256;
        d.strips = (N + d.strip - 1) / d.strip;
        const int64_t rest = N - (d.strips - 1) * d.strip;
        d.last = gemm16_plan(M, rest, K);
        d.full = rest == d.strip ? d.last : gemm16_plan(M, d.strip, K);
        d.us = (double)(d.strips - 1) * (d.full.us + 5.0) + d.last.us;
        d.weight_bytes = ((uint64_t)d.strip * (uint64_t)K * 2 + 255) / 256 * 256;
        const uint64_t pa = d.strips > 1 ? gemm16_part_bytes(d.full, M, d.strip) : 0, pb = gemm16_part_bytes(d.last, M, rest);
        d.part_bytes = pa > pb ? pa : pb;
        if (d.us < best.us) best = d;
        if (most >= N) break;
    }
    return best;
}
// What the many-rows streaming kernel takes, in us, fitted to 96 calls of 65 .. 2100 rows (median error 5 %): a workgroup of 128
// columns and R rows (64, 128, 192 or 256) walks 4096 k in DQ + 0.242 R beside 7.5 us a launch, where DQ is what dequantising takes;
// with 64 columns, where 64 rows leave the chip idle (use_cols64), 0.55 times that.  Rows as wq_narrow_slab_rows deals them, or
// in passes of 256.  With more than 128 rows and a K that is no whole number of x rounds of those instances, three times that;
// bf16 with 8-bit weights has no 256-row instance that fits and takes 1.6 times that there.
static double rows_kernel_us(const OpsnnWqmmArgs& a, int wbits, int64_t group)
{
    const int64_t wgs = (a.N + 127) / 128, kc = 4 * (128 / wbits), slab = wq_narrow_slab_rows(a.M, a.N, true);
    const int64_t ks = wq_rows_ksplit(wbits, a.M, a.N, a.K, group, true);
    const bool bf16 = a.x_dtype == DT_BF16, ragged = a.K % (8 * kc) != 0;
    const double dq = wq_rows_dequant_us(wbits, bf16);
    auto launch_us = [&](int64_t rows, int64_t slabs) {
        const int64_t r = (rows + 63) / 64 * 64, n = wgs * slabs * ks;
        const bool cols64 = r <= 64 && ks == 1 && wgs * slabs <= 128 && a.K % (4 * kc) == 0;
        const double rounds = cols64 ? 0.55 : n < 256 ? 0.94 + 0.06 * (double)n / 256.0 : (double)((n + 255) / 256);
        const double more = r > 128 && ragged ? 3.0 : r > 192 && bf16 && wbits == 8 ? 1.6 : 1.0;
        return 7.5 + rounds * (double)a.K / (4096.0 * (double)ks) * (dq + 0.242 * (double)r) * more;
    };
    const double part_us = ks > 1 ? 2.0 + 8.0 * (double)ks * (double)a.M * (double)a.N / 5.0e6 : 0.0;
    if (slab) return launch_us(slab, (a.M + slab - 1) / slab) + part_us;
    return (double)(a.M / 256) * launch_us(256, 1) + (a.M % 256 ? launch_us(a.M % 256, 1) : 0.0) + part_us;
}
// The tile kernel of wqmm_tile.hip, from 129 rows, in passes of up to 256 rows and workgroups of 128 columns.
static double tile_kernel_us(const OpsnnWqmmArgs& a, const WqForm& f)
{
    const double per = f.wbits == 8 ? 16.2 : f.group < 128 ? 15.6 : 14.65;
    return (double)((a.M + 255) / 256) * (6.0 + per * (double)a.K / 1024.0 * (double)((a.N + 32767) / 32768));
}

// Is this route faster than the kernel that would take the call otherwise?  The pass moves 2.5 (8-bit weights: 3) bytes per weight
// at 6 TB/s ([K, N] storage: 3.5, 4.6 with 8-bit weights), the product takes product_us (gemm16_plan) and 0.2 us more per 10^6
// weights, which it reads from beyond its L2.  Against it stand, with [K, N] storage behind a re-layout at 0.62 (0.73) TB/s of
// codes: the many-rows kernel where its shape conditions hold (with groups in [K, N] storage its scale table, and so its
// 192- and 256-row instances, do not apply); else, from 129 rows, the tile kernel and up to 128 rows the streaming kernel.
// With groups that are not whole chunks the general kernel is left, which counts where wq_general_counts says so.
// (The rule from 1025 rows on.  Of 368 calls of 65 .. 2100 rows, measured with the product's former plan, 362 go to the faster side or one within 3 % of it (profiles/weight_only_routes.txt): 1999 x 4096 x 11008
// bf16 x int4 228 -> 164 us, [K, N] storage 613 -> 162; 1000 x 8192 x 28672 fp16 x int4 stays on the many-rows kernel, 477 against 526; 65 x 4096 x 22896 on the streaming kernel, 54 against 93; 192 x 8192 x 22896 on the tile kernel, 127
// against 230; 128 x 11008 x 4096 in [K, N] storage with the re-layout, 61 against 75.)
struct DenseEstimate { double here, other; };
static DenseEstimate dense_estimate(const OpsnnWqmmArgs& a, double product_us)
{
    const WqForm f = wq_form(a);
    const double codes = (double)a.N * (double)a.K;
    double other;
    const bool four = f.wbits == 4, tile_ok = a.K % (four ? 128 : 64) == 0 && f.group % 64 == 0;
    const bool no_table = !f.nk && f.group < a.K;
    const double tile_us = tile_kernel_us(a, f) * (no_table ? 1.25 : 1.0);
    const double pass_rate = f.nk ? 6.0e6 : four ? 3.5e6 : 4.6e6;
    const double here = 3.0 + codes * (2.0 + f.wbits / 8.0) / pass_rate + product_us + codes * 2.0e-7;
    if (f.rows) {
        const int64_t slab = wq_narrow_slab_rows(a.M, a.N, true);
        if (no_table && (slab ? slab : a.M) > 128) other = tile_us;
        else other = rows_kernel_us(a, f.wbits, f.group) * (no_table && a.x_dtype == DT_BF16 ? 1.25 : 1.0);
    }
    else if (a.M > 128 && tile_ok) other = tile_us;
    else if (f.stream) other = wq_passes_of_64_us(a.M, [&](int64_t r) { return wq_stream_pass_us(f.wbits, a.x_dtype == DT_BF16, r, a.N, a.K); });
    else if (wq_general_counts(a, f)) other = wq_passes_of_64_us(a.M, [&](int64_t r) { return wq_general_pass_us(r, a.N, a.K); });
    else return {here, 1e30};
    if (!f.nk) other += 2.0 + codes * f.wbits / 8.0 / (four ? 0.62e6 : 0.73e6);
    return {here, other};
}
// The kernels of 33 rows and more on the terms of wq_cost.h.  The many-rows kernel up to 64 rows: its estimate as corrected by 396 calls (median error
// 4 %).
static double rows_typical_us(const OpsnnWqmmArgs& a, const WqForm& f)
{
    static const double rate[2][2] = {{1.19, 1.02}, {1.1, 1.1}}, offs[2][2] = {{0.03, 0.28}, {0.12, 0.11}};   // [8 bits][bf16]
    const int w8 = f.wbits == 8, bf = a.x_dtype == DT_BF16;
    return rows_kernel_us(a, f.wbits, f.group) * rate[w8][bf] * (a.offset ? 1.0 + offs[w8][bf] : 1.0) - 3.88 + 1.49e-6 * (double)a.M * (double)a.N;
}
// From 65 rows, to 1024: a workgroup of 128 columns and R rows as in rows_kernel_us, fitted to 340 calls (half of them for the fit, median error of the
// others 4 %).  Where the instance of 192 or 256 rows has no room for its table of scales beside x, or K is no multiple of 512, the call runs on the
// tile kernel: 682 x 12288 x 9856 int4 in groups of 128 takes 575 us there, 230 on the wide kernel.
static double many_rows_typical_us(const OpsnnWqmmArgs& a, const WqForm& f)
{
    static const double dq[2][2] = {{7.12, 10.9}, {11.6, 19.6}}, dq_off[2][2] = {{1.9, 9.4}, {4.9, 4.3}};          // [8 bits][bf16]
    static const double more[2][2][2] = {{{0.95, 1.04}, {0.85, 0.85}}, {{0.915, 0.937}, {1.03, 1.43}}};             // [more than 192 rows]: of R
    const int w8 = f.wbits == 8, bf = a.x_dtype == DT_BF16;
    const int64_t wgs = (a.N + 127) / 128, kc = 4 * (128 / f.wbits), slab = wq_narrow_slab_rows(a.M, a.N, true);
    const int64_t ks = wq_rows_ksplit(f.wbits, a.M, a.N, a.K, f.group, true), most = slab ? slab : a.M < 256 ? a.M : 256;
    if (most > 128) {
        int64_t pitch = 1;
        while (pitch * f.group < a.K) pitch *= 2;
        if (a.K % 512 != 0 || (most > 192 ? 131072 : 98304) + 512 * pitch > 163840) return tile_kernel_us(a, f);
    }
    const double cols = dq[w8][bf] + (a.offset ? dq_off[w8][bf] : 0.0), out_m = (double)a.M * (double)a.N * 1e-6;
    auto launch_us = [&](int64_t rows, int64_t slabs) {
        const int64_t r = (rows + 63) / 64 * 64, n = wgs * slabs * ks;
        const bool cols64 = r <= 64 && ks == 1 && wgs * slabs <= 128 && a.K % (4 * kc) == 0;
        const double rounds = cols64 ? 0.597 : (double)((n + 255) / 256);
        return 4.39 + rounds * (double)a.K / (4096.0 * (double)ks) * (cols + 0.173 * (double)r) * (r > 128 ? more[r > 192][w8][bf] : 1.0);
    };
    const double rest = 1.486 * out_m + (ks > 1 ? 2.0 + 3.41 * (double)ks * out_m : 0.0);
    if (slab) return launch_us(slab, (a.M + slab - 1) / slab) + rest;
    return (double)(a.M / 256) * launch_us(256, 1) + (a.M % 256 ? launch_us(a.M % 256, 1) : 0.0) + rest;
}
// The pass with its product, from 65 rows to 1024 (937 calls, half of them for the fit, 4 %).
static double dense_typical_us(const OpsnnWqmmArgs& a, const WqForm& f, double product_us)
{
    static const double pass[2][2] = {{0.3925, 0.4075}, {0.31, 0.336}};   // [K-contiguous][8 bits]: us per 10^6 codes
    const double codes = (double)a.N * (double)a.K * 1e-6;
    return 7.71 + codes * pass[f.nk][f.wbits == 8] * (1.0 + 0.578 * (codes < 200.0 ? codes / 100.0 : 2.0)) + 0.769 * product_us +
           0.704e-6 * (double)a.M * (double)a.N;
}
// Up to 1024 rows the typical times decide, as they do between this route and the wide kernel; beyond, the estimates above.  (With those for all
// of them, fitted to the product's former estimate, 558 x 1728 x 27136 bf16 x int8 went to the tile kernel, 85 -> 111 us.)
static bool dense_is_faster(const OpsnnWqmmArgs& a, double product_us)
{
    const DenseEstimate e = dense_estimate(a, product_us);
    if (a.M > 1024) return e.here < 0.97 * e.other;   // (in doubt without the pass)
    const WqForm f = wq_form(a);
    return dense_typical_us(a, f, product_us) < (f.rows && f.nk ? many_rows_typical_us(a, f) : e.other);
}
// What a call of 33 to 1024 rows typically takes without the wide kernel (wq_wide.hip), for its rule.
double wq_many_rows_typical_us(const OpsnnWqmmArgs& a)
{
    const WqForm f = wq_form(a);
    if (a.M <= 64) return f.rows && f.nk ? rows_typical_us(a, f) : 1e30;
    const double product_us = dense_plan(a.M, a.N, a.K).us;
    if (a.K % 64 == 0 && a.N >= 128 && dense_is_faster(a, product_us)) return dense_typical_us(a, f, product_us);
    return f.rows && f.nk ? many_rows_typical_us(a, f) : dense_estimate(a, product_us).other;
}

// Can the call run here?
static bool dense_takes(const OpsnnWqmmArgs& a, const WqForm& f)
{
    if (a.w_dtype != DT_I4 && a.w_dtype != DT_I8) return false;
    if (a.x_dtype != DT_F16 && a.x_dtype != DT_BF16) return false;
    if (a.scale_dtype != a.x_dtype || a.force_variant == OPSNN_VARIANT_PLAIN) return false;
    if (opsnn_wq_tile_min() <= 128) return false;   // (test hook: such calls are sent to the tile kernel of wqmm_tile.hip)
    if (a.M <= 64 || a.K % 64 != 0 || a.N < 128 || (uintptr_t)a.x % 16) return false;
    if (a.K >= (1ll << 22) || a.N >= (1ll << 24) || a.N * a.K >= (1ll << 36)) return false;   // (what the grids of the pass hold)
    if (a.group > 0 && a.group % 8 != 0) return false;
    if (!f.nk && (a.w.col_stride != 1 || a.w.row_stride != a.N)) return false;
    return a.w_dtype != DT_I4 || f.nk || a.N % 2 == 0;
}
// (K-contiguous outside the many-rows kernel's shapes: planned for in any case, since the other kernels take no weight at an
// unaligned address)
static bool always_planned(const WqForm& f) { return f.nk && !f.rows; }

// Workspace of this route, 0 if phase 1 does not plan for it.  Looks at what both phases know: shapes, types and layouts, not the
// weight's address.
uint64_t wq_dense_workspace(const OpsnnWqmmArgs& a)
{
    const WqForm f = wq_form(a);
    if (!dense_takes(a, f)) return 0;
    const DensePlan pl = dense_plan(a.M, a.N, a.K);
    if (!always_planned(f) && !dense_is_faster(a, pl.us)) return 0;
    return pl.weight_bytes + pl.part_bytes;
}

bool weight_cache_on();   // weight_cache.hip
const void* weight_cache_get(const void* src, int64_t K, int64_t N, int bits, int64_t nb, hipStream_t st);
int launch_wqmm_mfma(const OpsnnWqmmArgs& a, hipStream_t st);   // wqmm.hip

int launch_wq_dense(const OpsnnWqmmArgs& a, hipStream_t st)
{
    const WqForm f = wq_form(a);
    if (!a.workspace || !dense_takes(a, f)) return OPSNN_NOT_TAKEN;
    const int wbits = f.wbits;
    const bool kn = !f.nk, unaligned = (uintptr_t)a.w.ptr % 16 != 0;
    const DensePlan pl = dense_plan(a.M, a.N, a.K);
    if (!(always_planned(f) && unaligned) && !dense_is_faster(a, pl.us)) return OPSNN_NOT_TAKEN;
    if (kn && weight_cache_on()) {
        // a caller who keeps K-contiguous copies in the weight cache: where that form runs on another kernel, so does the copy
        // (128 x 8192 x 28672 int4: 75 us, 329 with the pass here); phase 1 has left room for its partial sums
        OpsnnWqmmArgs b = a;
        b.w.row_stride = 1; b.w.col_stride = a.K;
        if (!dense_is_faster(b, pl.us) && (b.w.ptr = weight_cache_get(a.w.ptr, a.K, a.N, wbits, 1, st)) != nullptr) {
            const int rc = launch_wqmm_mfma(b, st);
            if (rc != OPSNN_NOT_TAKEN) return rc;
        }
    }
    const bool two = pl.last.rows || pl.last.cols;   // (the product of the last strip, of all columns where there is one)
    note_route(two ? "wq_dense_two" : "wq_dense", two ? pl.last.rest_splits : pl.last.splits);
    uint16_t* w16 = (uint16_t*)a.workspace;
    WqParams p{};
    p.ldw = (kn ? a.w.row_stride : a.w.col_stride) * wbits / 8;
    p.s_rs = a.scale.row_stride; p.s_cs = a.scale_n == 1 ? 0 : a.scale.col_stride;
    p.M = a.M; p.K = a.K;
    p.group = a.group > 0 ? a.group : a.K;
    p.group_shift = (p.group & (p.group - 1)) == 0 ? __builtin_ctzll((unsigned long long)p.group) : p.group >= p.K ? 31 : -1;
    const bool f16 = a.x_dtype == DT_F16;
    const int bias_bytes = a.bias_dtype == DT_F32 ? 4 : 2;
    for (int64_t i = 0; i < pl.strips; i++) {
        const int64_t n0 = i * pl.strip;
        p.N = i + 1 < pl.strips ? pl.strip : a.N - n0;
        p.w = (const uint8_t*)a.w.ptr + (kn ? n0 * wbits / 8 : n0 * p.ldw);
        p.scale = (const uint16_t*)a.scale.ptr + n0 * p.s_cs;
        p.offset = a.offset ? (const uint16_t*)a.offset + n0 * p.s_cs : nullptr;
        int rc;
        if (f16) {
            if (wbits == 4) rc = a.offset ? launch_dequant<DT_F16, 4, true>(p, kn, w16, st) : launch_dequant<DT_F16, 4, false>(p, kn, w16, st);
            else rc = a.offset ? launch_dequant<DT_F16, 8, true>(p, kn, w16, st) : launch_dequant<DT_F16, 8, false>(p, kn, w16, st);
        } else {
            if (wbits == 4) rc = a.offset ? launch_dequant<DT_BF16, 4, true>(p, kn, w16, st) : launch_dequant<DT_BF16, 4, false>(p, kn, w16, st);
            else rc = a.offset ? launch_dequant<DT_BF16, 8, true>(p, kn, w16, st) : launch_dequant<DT_BF16, 8, false>(p, kn, w16, st);
        }
        if (rc != 0) return rc;
        QgemmParams g{};
        g.a = (const int8_t*)a.x; g.b = (const int8_t*)w16;
        g.lda = 2 * a.K; g.ldb = 2 * a.K; g.KB = 2 * a.K;
        g.out = (uint16_t*)a.y + n0; g.M = a.M; g.N = p.N; g.ldc = a.N;
        g.bias = a.bias ? (const char*)a.bias + n0 * bias_bytes : nullptr; g.bias_dt = a.bias_dtype;
        rc = launch_gemm16(g, i + 1 < pl.strips ? pl.full : pl.last, !f16, (float*)((char*)a.workspace + pl.weight_bytes), st);
        if (rc != 0) return rc;
    }
    return 0;
}

}  // namespace opsnn
