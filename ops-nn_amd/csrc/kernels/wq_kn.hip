// Weight-only matmul with few rows of x (up to 64) against a weight in its [K, N] storage: the weight is streamed once, as it
// lies.  (It was re-laid out K-contiguous in front of the streaming kernels on every call: 16 x 8192 x 28672 int4 245 us, of which
// that pass 214.)
//
// The k order inside a matrix instruction is free as long as both operands agree, and so is which output column a row of
// the weight operand stands for.  A lane (r = lane % 16, q = lane / 16) loads CPL neighbouring codes of the 8 rows
// k = 8 q .. 8 q + 7 of a 32-k step: 16 lanes side by side make 128 contiguous bytes of a weight row (int4, 16 codes per
// lane; int8 256).  Dequantised along the columns and transposed 8 x 8 in registers (dequant_8x8), every one of its CPL
// columns becomes 8 consecutive k: the operand of one v_mfma_f32_16x16x32 whose row r is column n0 + CPL r + c.  x is the
// other operand straight from memory (16 bytes per lane and 16 rows; it stays in L2).  No LDS in the loop, no barrier.
//
// The loads of a step are held or in flight while others multiply, which the compiler's waits have to see: with conditions on the fetches
// and on the scales it waits for every load under way in each step.  From some twelve steps a wave (TABLE, up to 16 rows) the loop has
// none: the fetches go on past the end, and the scales of a window of steps lie in LDS (16 x 8192 x 28672 int4 44.4 -> 40.7 us, 3 x 11904 x 21504
// 41.4 -> 38.2).
//
// Work split: a workgroup is four waves on the same 16 CPL columns, each with a quarter of the workgroup's steps; blockIdx.y
// cuts K into segments so that the chip has two workgroups per CU.  With the table and an even count of segments, two of them are one workgroup of
// eight waves, which halves the partial sums (16 x 8192 x 28672 42.0 -> 40.4 us, 9 x 12032 x 19648 43.9 -> 42.5, int8 10 x 15616 x 12352 47.3 -> 45.6).  The waves' sums meet in LDS in a fixed order; with more
// than one segment they go to `part` as fp32 and wq_splitk_reduce_kernel adds the segments in order.
#include "launch.h"
#include "wq_cost.h"
#include "wq_kn.hip.h"
#include "wqmm_stream.hip.h"

namespace opsnn {

struct WqKnPlan {
    int mb = 1, splits = 1;
};
constexpr int KN_GROUPS = 16;   // groups in a wave's table of scales
constexpr int kn_pf(int wbits, int mb) { return (mb == 2 || (mb == 1 && wbits == 4)) ? 3 : 2; }   // steps held or in flight per wave
constexpr int kn_cpl(int mb) { return mb == 1 ? 16 : 8; }   // codes per lane: with 16 and two row blocks the loop spills

// Segments of K: as many workgroups as two per CU, less what a slice of partial sums costs.  (A step is 4 KB (int8: 8 KB) per
// wave; at 5 TB/s the eight waves of a CU take 1.7 us for one each.  3 us: the second kernel.  Segments that run in pairs on eight waves
// (launch_kn_mb) are priced one by one, which charges them for partial sums that they don't write.  Of 40 calls 35 run within 3 % of the
// fastest count, the worst 5.5 % behind: 64 x 2048 x 16384 24.2 us, 22.9 with two segments; profiles/tile_plans.txt.  512: two
// workgroups on each of the chip's 256 CUs, a constant, since phase 1 plans too and makes no HIP call.)
static WqKnPlan kn_plan(int wbits, int64_t M, int64_t N, int64_t K)
{
    WqKnPlan pl;
    pl.mb = M <= 16 ? 1 : M <= 32 ? 2 : 4;
    const int64_t strips = (N + 16 * kn_cpl(pl.mb) - 1) / (16 * kn_cpl(pl.mb)), steps = K / 32;
    const double t_step = (pl.mb == 4 ? 1.4 : pl.mb == 2 ? 1.0 : 1.7) * (wbits == 8 ? 1.8 : 1.0);
    double best = 1e30;
    for (int s = 1; s <= 16 && steps / s >= 8; s++) {
        const double us = (double)((strips * s + 511) / 512) * ((double)((steps + 4 * s - 1) / (4 * s)) * t_step + 3.0) +
                          (s > 1 ? 3.0 + 8.0 * s * (double)M * (double)N / 4.0e6 : 0.0);
        if (us < best) { best = us; pl.splits = s; }
    }
    return pl;
}

template <int XDT, int WBITS, int MB, bool HAS_OFF, bool TABLE, int NW>
__global__ __launch_bounds__(64 * NW, 8 / NW) void wq_kn_kernel(WqParams p, int splits, int window)
{
    constexpr int CPL = kn_cpl(MB);
    constexpr int DW = CPL * WBITS / 32;          // dwords of codes per lane and row: 1, 2 or 4
    constexpr int OCT = CPL / 8;                  // 8 x 8 blocks per step
    constexpr int PF = kn_pf(WBITS, MB);
    extern __shared__ __attribute__((aligned(16))) float red[];   // two waves' sums
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, q = lane >> 4;
    const int64_t strip0 = (int64_t)blockIdx.x * (16 * CPL);
    // this lane's first column; past the edge of the matrix the last CPL columns again (computed twice, stored once)
    const int64_t nl = strip0 + r * CPL, n = nl + CPL <= p.N ? nl : p.N - CPL;
    const int steps = (int)(p.K / 32);
    const int s0 = (int)((int64_t)blockIdx.y * steps / splits), s1 = (int)((int64_t)(blockIdx.y + 1) * steps / splits);
    const int w0 = s0 + (s1 - s0) * wave / NW, w1 = s0 + (s1 - s0) * (wave + 1) / NW;   // this wave's steps

    const uint8_t* wbase = p.w + (int64_t)8 * q * p.ldw + n * WBITS / 8;
    const int64_t ldw = p.ldw;
    const uint16_t* sbase = p.scale + n * p.s_cs;
    const uint16_t* obase = HAS_OFF ? p.offset + n * p.s_cs : nullptr;
    const uint16_t* xrow[MB];
#pragma unroll
    for (int b = 0; b < MB; b++) {
        const int64_t m = 16 * b + r;
        xrow[b] = p.x + (m < p.M ? m : p.M - 1) * p.K + 8 * q;
    }
    const int groupi = (int)p.group;
    auto group_of = [&](int st) { return p.group_shift >= 0 ? (st * 32) >> p.group_shift : (st * 32) / groupi; };

    v4f acc[CPL][MB];
#pragma unroll
    for (int c = 0; c < CPL; c++)
#pragma unroll
        for (int b = 0; b < MB; b++) acc[c][b] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
    auto multiply = [&](const uint32_t (&rw)[8][DW], const v4i (&x)[MB], const uint32_t (&sc)[OCT][4], const uint32_t (&of)[OCT][4]) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < OCT; t++) {
            uint32_t q8[8][WBITS / 4], o[8][4];
#pragma unroll
            for (int i = 0; i < 8; i++)
#pragma unroll
                for (int d = 0; d < WBITS / 4; d++) q8[i][d] = rw[i][t * (WBITS / 4) + d];
            dequant_8x8<XDT, WBITS, HAS_OFF>(q8, sc[t], of[t], o);
#pragma unroll
            for (int c = 0; c < 8; c++) {
                const v4i a = {(int)o[c][0], (int)o[c][1], (int)o[c][2], (int)o[c][3]};
#pragma unroll
                for (int b = 0; b < MB; b++) {
                    v4f& d = acc[t * 8 + c][b];
                    if constexpr (XDT == DT_F16) d = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, x[b]), d, 0, 0, 0);
                    else d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, x[b]), d, 0, 0, 0);
                }
            }
        }
    };
    if constexpr (TABLE) {
        uint32_t raw[PF][8][DW];
        v4i xf[PF][MB];
        auto fetch = [&](auto jc, int st) {   // (past the end: the last step again, so that every step waits for the same count of loads)
            constexpr int j = decltype(jc)::value;
            const int sc = st < w1 ? st : w1 - 1;
            const uint8_t* w = wbase + (int64_t)sc * 32 * ldw;
#pragma unroll
            for (int i = 0; i < 8; i++) __builtin_memcpy(raw[j][i], w + i * ldw, 4 * DW);
#pragma unroll
            for (int b = 0; b < MB; b++) xf[j][b] = *(const v4i*)(xrow[b] + sc * 32);
            __builtin_amdgcn_sched_barrier(0);
        };

        // scales of a window of steps: rows of 16 CPL columns, this wave's own
        char* const tab = (char*)red + wave * (KN_GROUPS * 32 * CPL * (HAS_OFF ? 2 : 1));
        int g_lo = 0;
        auto load_window = [&](int st, int end) {
            g_lo = group_of(st);
            const int n_groups = group_of(end - 1) - g_lo + 1;
            wave_lds_fence();   // (other lanes of the wave read what a lane writes here, and read the window before until now)
            for (int g = q; g < n_groups; g += 4) {   // (lane r: its own CPL columns)
                uint32_t v[HAS_OFF ? 2 : 1][CPL / 2];
                if (p.s_cs == 1) {
                    __builtin_memcpy(v[0], sbase + (int64_t)(g_lo + g) * p.s_rs, 2 * CPL);
                    if constexpr (HAS_OFF) __builtin_memcpy(v[1], obase + (int64_t)(g_lo + g) * p.s_rs, 2 * CPL);
                } else {   // one scale for all columns (s_cs == 0)
#pragma unroll
                    for (int e = 0; e < CPL / 2; e++) {
                        v[0][e] = sbase[(int64_t)(g_lo + g) * p.s_rs] * 0x00010001u;
                        if constexpr (HAS_OFF) v[1][e] = obase[(int64_t)(g_lo + g) * p.s_rs] * 0x00010001u;
                    }
                }
                __builtin_memcpy(tab + g * (32 * CPL) + r * (2 * CPL), v[0], 2 * CPL);
                if constexpr (HAS_OFF) __builtin_memcpy(tab + (KN_GROUPS + g) * (32 * CPL) + r * (2 * CPL), v[1], 2 * CPL);
            }
            wave_lds_fence();
        };
        auto step = [&](auto jc, int st) __attribute__((always_inline)) {
            constexpr int j = decltype(jc)::value;
            const char* const at = tab + (group_of(st) - g_lo) * (32 * CPL) + r * (2 * CPL);
            uint32_t sc[OCT][4], of[OCT][4] = {};
            __builtin_memcpy(sc, __builtin_assume_aligned(at, 16), sizeof(sc));
            if constexpr (HAS_OFF) __builtin_memcpy(of, __builtin_assume_aligned(at + KN_GROUPS * (32 * CPL), 16), sizeof(of));
            multiply(raw[j], xf[j], sc, of);
            __builtin_amdgcn_sched_barrier(0);
        };
        auto each = [&](auto&& f) {
            [&]<int... J>(std::integer_sequence<int, J...>) { (f(std::integral_constant<int, J>{}), ...); }(std::make_integer_sequence<int, PF>{});
        };
        if (w0 < w1) {
            each([&](auto j) { fetch(j, w0 + j); });
            int st = w0;
            while (w1 - st >= PF) {   // windows of whole rounds of PF steps
                int end = w1 - st > window ? st + window : st + (w1 - st) / PF * PF;
                load_window(st, end);
                for (; st < end; st += PF) each([&](auto j) __attribute__((always_inline)) { step(j, st + j); fetch(j, st + j + PF); });
            }
            if (st < w1) {
                load_window(st, w1);
                each([&](auto j) __attribute__((always_inline)) { if (st + j < w1) step(j, st + j); });
            }
        }
        __syncthreads();   // the tables make room for the sums
    } else {
        uint32_t raw[PF][8][DW];
        v4i xf[PF][MB];
        uint32_t sc[OCT][4], of[OCT][4];
#pragma unroll
        for (int t = 0; t < OCT; t++)
#pragma unroll
            for (int e = 0; e < 4; e++) sc[t][e] = of[t][e] = 0;
        auto fetch = [&](auto jc, int st) {
            constexpr int j = decltype(jc)::value;
            const uint8_t* w = wbase + (int64_t)st * 32 * ldw;
#pragma unroll
            for (int i = 0; i < 8; i++) __builtin_memcpy(raw[j][i], w + i * ldw, 4 * DW);
#pragma unroll
            for (int b = 0; b < MB; b++) xf[j][b] = *(const v4i*)(xrow[b] + st * 32);
        };
        auto load_scales = [&](int g) {
            if (p.s_cs == 1) {
                __builtin_memcpy(sc, sbase + (int64_t)g * p.s_rs, sizeof(sc));
                if constexpr (HAS_OFF) __builtin_memcpy(of, obase + (int64_t)g * p.s_rs, sizeof(of));
            } else {   // one scale for all columns (s_cs == 0)
#pragma unroll
                for (int t = 0; t < OCT; t++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        sc[t][e] = sbase[(int64_t)g * p.s_rs] * 0x00010001u;
                        if constexpr (HAS_OFF) of[t][e] = obase[(int64_t)g * p.s_rs] * 0x00010001u;
                    }
            }
        };

        int g_cur = -1;
        auto step = [&](auto jc, int st) {
            constexpr int j = decltype(jc)::value;
            const int g = group_of(st);
            if (g != g_cur) { load_scales(g); g_cur = g; }
            multiply(raw[j], xf[j], sc, of);
            if (st + PF < w1) fetch(jc, st + PF);
        };
        using I0 = std::integral_constant<int, 0>;
        using I1 = std::integral_constant<int, 1>;
        using I2 = std::integral_constant<int, PF - 1>;
        if (w0 < w1) fetch(I0{}, w0);
        if (w0 + 1 < w1) fetch(I1{}, w0 + 1);
        if constexpr (PF == 3) { if (w0 + 2 < w1) fetch(I2{}, w0 + 2); }
        for (int st = w0; st < w1; st += PF) {
            step(I0{}, st);
            if (st + 1 < w1) step(I1{}, st + 1);
            if constexpr (PF == 3) { if (st + 2 < w1) step(I2{}, st + 2); }
        }
    }

    if (!sum_of_waves<NW>(acc, red, wave, lane)) return;

    // acc[c][b][i] is out[m = 16 b + lane % 16][column c of the weight rows' lane 4 q + i]: CPL neighbouring columns per i
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int64_t ns = strip0 + (4 * q + i) * CPL;
        if (ns >= p.N) continue;
        const int64_t nn = ns + CPL <= p.N ? ns : p.N - CPL;
#pragma unroll
        for (int b = 0; b < MB; b++) {
            const int64_t m = 16 * b + r;
            if (m >= p.M) continue;
            if (splits > 1) {
                float* dst = p.part + ((int64_t)blockIdx.y * p.M + m) * p.N + nn;
#pragma unroll
                for (int c = 0; c < CPL; c += 4) {
                    const v4f v = {acc[c][b][i], acc[c + 1][b][i], acc[c + 2][b][i], acc[c + 3][b][i]};
                    __builtin_memcpy(dst + c, &v, 16);
                }
            } else {
                uint16_t* dst = p.y + m * p.N + nn;
#pragma unroll
                for (int c = 0; c < CPL; c += 4) {
                    uint16_t o[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        float v = acc[c + e][b][i];
                        if (p.bias) v = v + load_scalar_as_f32(p.bias, p.bias_dt, nn + c + e);
                        o[e] = bits_x<XDT>(v);
                    }
                    __builtin_memcpy(dst + c, o, 8);
                }
            }
        }
    }
}

template <int XDT, int WBITS, int MB, bool HAS_OFF, bool TABLE = false, int NW = 4>
static int launch_kn_one(const WqParams& p, int splits, hipStream_t st)
{
    constexpr int CPL = kn_cpl(MB), PF = kn_pf(WBITS, MB);
    const dim3 grid((unsigned)((p.N + 16 * CPL - 1) / (16 * CPL)), (unsigned)splits);
    constexpr size_t lds_sum = (size_t)NW / 2 * CPL * MB * 4 * 64 * 4, lds_tab = TABLE ? (size_t)NW * KN_GROUPS * 32 * CPL * (HAS_OFF ? 2 : 1) : 0;
    constexpr size_t lds = lds_sum > lds_tab ? lds_sum : lds_tab;
    // steps whose groups fit a table wherever they start, in whole rounds of the loop
    const int64_t steps = p.K / 32, fit = p.group >= p.K ? steps + PF : (KN_GROUPS - (p.group > 32)) * p.group / 32;
    const int window = (int)((fit < steps + PF ? fit : steps + PF) / PF * PF);
    auto k = wq_kn_kernel<XDT, WBITS, MB, HAS_OFF, TABLE, NW>;
    static std::atomic<uint64_t> attr_set{0};   // one bit per device: the attribute belongs to the (kernel, device) pair
    if (!device_flag_test(attr_set)) {
        hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return (int)e;
        device_flag_set(attr_set);
    }
    note_route(NW == 8 ? "wq_kn_table_w8" : TABLE ? "wq_kn_table" : "wq_kn", splits);
    hipLaunchKernelGGL(k, grid, dim3(64 * NW), lds, st, p, splits, window);
    if (hipError_t e = hipGetLastError(); e != hipSuccess || splits == 1) return (int)e;
    launch_wq_splitk_reduce(p, splits, XDT, st);
    return (int)hipGetLastError();
}
template <int XDT, int WBITS, bool HAS_OFF>
static int launch_kn_mb(const WqParams& p, const WqKnPlan& pl, hipStream_t st)
{
    if (pl.mb == 1) {
        // (the table pays for itself from some twelve steps a wave: 16 x 8192 x 28672, sixteen, 44.4 -> 41.3 us; 4 x 3072 x 1872, six, 9.0 -> 10.4)
        if (p.K / 32 >= 48 * pl.splits && pl.splits % 2 == 0) return launch_kn_one<XDT, WBITS, 1, HAS_OFF, true, 8>(p, pl.splits / 2, st);
        if (p.K / 32 >= 48 * pl.splits) return launch_kn_one<XDT, WBITS, 1, HAS_OFF, true>(p, pl.splits, st);
        return launch_kn_one<XDT, WBITS, 1, HAS_OFF>(p, pl.splits, st);
    }
    if (pl.mb == 2) return launch_kn_one<XDT, WBITS, 2, HAS_OFF>(p, pl.splits, st);
    return launch_kn_one<XDT, WBITS, 4, HAS_OFF>(p, pl.splits, st);
}

bool weight_cache_on();   // weight_cache.hip

// Can the call run here?  Looks at what phase 1 knows, so that both phases agree.
bool wq_kn_wanted(const OpsnnWqmmArgs& a)
{
    if ((a.w_dtype != DT_I4 && a.w_dtype != DT_I8) || (a.x_dtype != DT_F16 && a.x_dtype != DT_BF16)) return false;
    if (a.scale_dtype != a.x_dtype || a.force_variant != 0) return false;
    if (a.M > 64 || a.K % 32 != 0 || a.K < 256 || a.N < 256 || a.K >= (1ll << 30) || a.N >= (1ll << 30)) return false;
    if (a.w.col_stride != 1 || a.w.row_stride != a.N || (a.w_dtype == DT_I4 && a.N % 2 != 0)) return false;
    if (a.group > 0 && a.group < a.K && a.group % 32 != 0) return false;
    // (so small a weight is re-laid out as fast -- 16 x 1024 x 512 9.7 us that way, 10.2 here -- and then gives the bits of its
    // pre-packed form)
    if (a.K * a.N < (1ll << 20)) return false;
    // (Up to 16 rows of 8-bit weights of at most 2^24 codes: slower on purpose.  16 x 4096 x 4096 int8 takes 28 us behind the
    // re-layout and 13 here, but the x-in-registers kernel behind it gives the bits of the [N, K] form, which callers at these sizes
    // have always had and the full-size tests assert.  Elsewhere the two storage forms agree to the summation order only.)
    if (a.w_dtype == DT_I8 && a.M <= 16 && a.K * a.N <= (1ll << 24)) return false;
    if (a.scale_n != 1 && a.scale.col_stride != 1) return false;
    return (uintptr_t)a.x % 16 == 0;
}
// What the kernel typically takes for a call that wq_kn_wanted accepts, for the rule of wq_wide.hip (592 calls, median error 4 %): us per
// step of a wave by row blocks.
double wq_kn_typical_us(const OpsnnWqmmArgs& a)
{
    static const double step[2][2][3] = {{{1.22, 0.85, 1.33}, {1.51, 0.89, 1.31}}, {{1.43, 0.86, 1.58}, {1.6, 0.93, 1.51}}};   // [8 bits][bf16]
    const int wbits = a.w_dtype == DT_I4 ? 4 : 8;
    const bool bf16 = a.x_dtype == DT_BF16;
    const WqKnPlan pl = kn_plan(wbits, a.M, a.N, a.K);
    const int64_t cols = 16 * kn_cpl(pl.mb), per_wave = (a.K / 32 + 4 * pl.splits - 1) / (4 * pl.splits);
    const double t = step[wbits == 8][bf16][pl.mb == 4 ? 2 : pl.mb - 1] + (a.offset ? (bf16 ? 0.46 : 0.18) : 0.0);
    const double cu = wq_typical_turns((a.N + cols - 1) / cols * pl.splits, 1.33) * ((double)per_wave * t + 1.7);
    return 4.5 + wq_typical_both(cu, wq_typical_mb(wbits, a.N, a.K) / 5.44) +
           (pl.splits > 1 ? 3.25e-6 * (double)pl.splits * (double)a.M * (double)a.N * (a.N % 4 ? 2.0 : 1.0) : 0.0);
}
uint64_t wq_kn_workspace(const OpsnnWqmmArgs& a)
{
    const WqKnPlan pl = kn_plan(a.w_dtype == DT_I4 ? 4 : 8, a.M, a.N, a.K);
    return pl.splits > 1 ? ((uint64_t)pl.splits * (uint64_t)a.M * (uint64_t)a.N * 4 + 255) / 256 * 256 : 0;
}
int launch_wq_kn(const OpsnnWqmmArgs& a, hipStream_t st)
{
    // (a caller who keeps K-contiguous copies in the weight cache has paid for them: those calls go on to the other kernels,
    // and phase 1 plans for either)
    if (!wq_kn_wanted(a) || weight_cache_on()) return OPSNN_NOT_TAKEN;
    const int wbits = a.w_dtype == DT_I4 ? 4 : 8;
    WqKnPlan pl = kn_plan(wbits, a.M, a.N, a.K);
    if (!a.workspace) pl.splits = 1;   // no room for partial sums: K in one piece
    WqParams p{};
    p.x = (const uint16_t*)a.x;
    p.w = (const uint8_t*)a.w.ptr; p.ldw = a.w.row_stride * wbits / 8;
    p.scale = (const uint16_t*)a.scale.ptr; p.offset = (const uint16_t*)a.offset;
    p.s_rs = a.scale.row_stride; p.s_cs = a.scale_n == 1 ? 0 : 1;
    p.bias = a.bias; p.bias_dt = a.bias_dtype;
    p.y = (uint16_t*)a.y; p.M = a.M; p.N = a.N; p.K = a.K;
    p.group = a.group > 0 ? a.group : a.K;
    p.group_shift = p.group >= p.K ? 31 : (p.group & (p.group - 1)) == 0 ? __builtin_ctzll((unsigned long long)p.group) : -1;
    p.part = (float*)a.workspace;
    if (a.x_dtype == DT_F16) {
        if (wbits == 4) return a.offset ? launch_kn_mb<DT_F16, 4, true>(p, pl, st) : launch_kn_mb<DT_F16, 4, false>(p, pl, st);
        return a.offset ? launch_kn_mb<DT_F16, 8, true>(p, pl, st) : launch_kn_mb<DT_F16, 8, false>(p, pl, st);
    }
    if (wbits == 4) return a.offset ? launch_kn_mb<DT_BF16, 4, true>(p, pl, st) : launch_kn_mb<DT_BF16, 4, false>(p, pl, st);
    return a.offset ? launch_kn_mb<DT_BF16, 8, true>(p, pl, st) : launch_kn_mb<DT_BF16, 8, false>(p, pl, st);
}

}  // namespace opsnn
