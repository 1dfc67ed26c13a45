// Weight-only matmul with few rows of x (up to 64) against a weight in [N, K] storage whose shape the specialised streaming
// kernels of wqmm_stream.hip.h do not take: any N, K a multiple of 32 (8-bit weights: 16 would do), any group that is a multiple
// of 32.  (Such calls -- N no multiple of 32, groups of 64, K % 128 = 64 -- ran on the general kernel: 17 x 5632 x 1453 49 us,
// 3 x 16448 x 2560 131 us.)
//
// A wave owns NB blocks of 16 columns; lane (r = lane % 16, q = lane / 16) streams PB-byte pieces of the rows 16 j + r straight
// into registers (32 int4 or 16 int8 with 16 bytes; 16 int4 with 8), two chunks ahead, and the pieces of x that go with them
// straight from memory: with eight (four) column blocks per x fragment the fragments cost no more requests than the weights, so
// there is no LDS and no barrier in the loop.  Scales and offsets lie in a table in LDS, one word per column and group, laid
// down once per workgroup (fetched per chunk they are 2-byte gathers of 16 cache lines each, as many requests as the weights).
// x is put into the order in which the nibble splice delivers the weights (one permute per register of x, shared by the
// column blocks).
//
// Work split as in wq_kn.hip: the four waves of a workgroup take a quarter each of its chunks, blockIdx.y cuts K into
// segments; sums meet in LDS in a fixed order, segments in `part`, added in order by wq_splitk_reduce_kernel.  A wave past the
// edge of N repeats the last columns (stored twice, same bits).
#include "launch.h"
#include "wq_cost.h"
#include "wqmm_stream.hip.h"

extern "C" int opsnn_wq_narrow_slabs();   // dispatch.hip
namespace opsnn {

struct WqNkPlan {
    int mb = 1, splits = 1;
    int groups = 1;   // groups a workgroup's segment can touch: columns of its scale table
};
// column blocks of 16 per workgroup (with four row blocks of x: sums, x fragments and eight column blocks would not fit the registers)
constexpr int nk_nb(int mb) { return mb == 4 ? 4 : 8; }
static bool nk_plan(int wbits, int64_t M, int64_t N, int64_t K, int64_t group, WqNkPlan& pl)
{
    pl.mb = M <= 16 ? 1 : M <= 32 ? 2 : 4;
    // (32-bit: both phases of every call with few rows come here; N and K are below 2^30.  512 below: two workgroups on each of the
    // chip's 256 CUs, a constant, since phase 1 makes no HIP call)
    const uint32_t cols = 16 * nk_nb(pl.mb), strips = ((uint32_t)N + cols - 1) / cols, kc = (pl.mb == 4 || wbits == 8) ? 64 : 128;
    const uint32_t chunks = ((uint32_t)K + kc - 1) / kc;
    // (a chunk: 8 KB of codes per wave; four row blocks: 2 KB of 4-bit, 4 KB of 8-bit codes; eight waves of a CU at 5 TB/s.  Of 24
    // calls 22 run within 10 % of the fastest count of segments; the worst, 16 x 8224 x 16384 int8, takes 54.6 us with its four and
    // 40.8 with two: profiles/tile_plans.txt)
    const double t_chunk = pl.mb == 4 ? (wbits == 4 ? 1.4 : 2.0) : pl.mb == 2 ? 4.1 : 3.4;
    const double slice_us = 8.0 * (double)M * (double)N / 4.0e6;
    double best = 1e30;
    bool found = false;
    for (uint32_t s = 1; s <= 16 && chunks >= 2 * s; s++) {
        const uint32_t seg = (chunks + s - 1) / s * kc, per_wave = (chunks + 4 * s - 1) / (4 * s);
        const uint32_t g = group >= K ? 1 : (seg + (uint32_t)group - 1) / (uint32_t)group + 1;
        if (g <= 8192 / cols) {   // (a table of 32 KB)
            const double us = (double)((strips * s + 511) / 512) * ((double)per_wave * t_chunk + 4.0) + (s > 1 ? 3.0 + slice_us * s : 0.0);
            if (us < best) { best = us; pl.splits = (int)s; pl.groups = (int)g; found = true; }
        }
        if (per_wave == 1 && found) break;   // (more segments only add partial sums)
    }
    return found;
}

template <int XDT, int WBITS, int MB, bool HAS_OFF>
__global__ __launch_bounds__(256, 2) void wq_nk_kernel(WqParams p, int splits, int gmax)
{
    constexpr int NB = nk_nb(MB), PF = 2;
    constexpr int PB = (MB == 4 && WBITS == 4) ? 8 : 16;   // bytes of a lane's weight piece
    constexpr int KPL = PB * 8 / WBITS, KC = 4 * KPL, STEPS = KPL / 8;
    constexpr int DW = PB / 4;
    extern __shared__ __attribute__((aligned(16))) float dyn[];   // the scale table; at the end two waves' sums
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, q = lane >> 4;
    int64_t n0 = (int64_t)blockIdx.x * (16 * NB);
    if (n0 + 16 * NB > p.N) n0 = p.N - 16 * NB;
    const int Ki = (int)p.K, chunks = (Ki + KC - 1) / KC;
    const int s0 = (int)((int64_t)blockIdx.y * chunks / splits), s1 = (int)((int64_t)(blockIdx.y + 1) * chunks / splits);
    const int w0 = s0 + (s1 - s0) * wave / 4, w1 = s0 + (s1 - s0) * (wave + 1) / 4;   // this wave's chunks

    // scale table: word (column, group - g_lo) = scale | offset << 16
    const int groupi = (int)p.group;
    auto group_at = [&](int k) { return p.group_shift >= 0 ? k >> p.group_shift : k / groupi; };
    const int g_lo = group_at(s0 * KC), g_all = group_at(Ki - 1);
    uint32_t* const tab = (uint32_t*)dyn;
    for (int i = tid; i < 16 * NB * gmax; i += 256) {
        const int col = i / gmax, gi = g_lo + i - col * gmax;
        const int64_t at = (int64_t)(gi < g_all ? gi : g_all) * p.s_rs + (n0 + col) * p.s_cs;
        uint32_t w = p.scale[at];
        if constexpr (HAS_OFF) w |= (uint32_t)p.offset[at] << 16;
        tab[col * gmax + i - col * gmax] = w;
    }
    __syncthreads();

    const uint8_t* wbase = p.w + (n0 + r) * p.ldw;
    const int64_t wblk = 16 * p.ldw;
    const uint16_t* xrow[MB];
#pragma unroll
    for (int b = 0; b < MB; b++) {
        const int64_t m = 16 * b + r;
        xrow[b] = p.x + (m < p.M ? m : p.M - 1) * p.K;
    }
    uint32_t raw[PF][NB][DW];
    v4i xf[PF][STEPS][MB];
    auto fetch = [&](auto jc, int c) {
        constexpr int j = decltype(jc)::value;
        const int k0 = c * KC + q * KPL, k = k0 < Ki ? k0 : Ki - KPL;   // (past the end of K: the last piece, which counts as zero)
        const uint8_t* w = wbase + (int64_t)k * WBITS / 8;
#pragma unroll
        for (int b = 0; b < NB; b++) __builtin_memcpy(raw[j][b], w + b * wblk, PB);
#pragma unroll
        for (int s = 0; s < STEPS; s++)
#pragma unroll
            for (int b = 0; b < MB; b++) xf[j][s][b] = *(const v4i*)(xrow[b] + k + 8 * s);
    };
    v4f acc[NB][MB];
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
        for (int b = 0; b < MB; b++) acc[j][b] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
    const DqConst dqc = make_dq_const();
    auto chunk = [&](auto jc, int c) {
        constexpr int j = decltype(jc)::value;
        const int k = c * KC + q * KPL;
        const int gi = group_at(k < Ki ? k : Ki - KPL) - g_lo;
        uint32_t sow[NB];
#pragma unroll
        for (int b = 0; b < NB; b++) sow[b] = tab[(16 * b + r) * gmax + gi];
        if (c == chunks - 1 && k >= Ki) {   // past the end of K: both factors zero (0 * inf is no zero; a code's weight is, with scale and offset 0)
#pragma unroll
            for (int s = 0; s < STEPS; s++)
#pragma unroll
                for (int b = 0; b < MB; b++) xf[j][s][b] = (v4i){0, 0, 0, 0};
#pragma unroll
            for (int b = 0; b < NB; b++) sow[b] = 0;
        }
#pragma unroll
        for (int s = 0; s < STEPS; s++) {
            v4i xo[MB];
#pragma unroll
            for (int b = 0; b < MB; b++) {
                xo[b] = xf[j][s][b];
                if constexpr (WBITS == 4) {   // halves [0..7] -> [0,4,1,5,2,6,3,7]
                    const uint32_t a0 = (uint32_t)xo[b][0], a1 = (uint32_t)xo[b][1], a2 = (uint32_t)xo[b][2], a3 = (uint32_t)xo[b][3];
                    xo[b] = (v4i){(int)__builtin_amdgcn_perm(a2, a0, 0x05040100u), (int)__builtin_amdgcn_perm(a2, a0, 0x07060302u),
                                  (int)__builtin_amdgcn_perm(a3, a1, 0x05040100u), (int)__builtin_amdgcn_perm(a3, a1, 0x07060302u)};
                }
            }
#pragma unroll
            for (int nb = 0; nb < NB; nb++) {
                v4i piece = {0, 0, 0, 0};
                if constexpr (WBITS == 4) piece[0] = (int)raw[j][nb][s];
                else { piece[0] = (int)raw[j][nb][2 * s]; piece[1] = (int)raw[j][nb][2 * s + 1]; }
                const v4i a = dequant8<XDT, WBITS, HAS_OFF>(piece, 0, (uint16_t)sow[nb], (uint16_t)(sow[nb] >> 16), dqc);
#pragma unroll
                for (int b = 0; b < MB; b++) {
                    if constexpr (XDT == DT_F16) acc[nb][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, xo[b]), acc[nb][b], 0, 0, 0);
                    else acc[nb][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, xo[b]), acc[nb][b], 0, 0, 0);
                }
            }
        }
        if (c + PF < w1) fetch(jc, c + PF);
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    if (w0 < w1) fetch(I0{}, w0);
    if (w0 + 1 < w1) fetch(I1{}, w0 + 1);
    for (int c = w0; c < w1; c += PF) {
        chunk(I0{}, c);
        if (c + 1 < w1) chunk(I1{}, c + 1);
    }

    __syncthreads();   // the scale table makes room
    if (!sum_of_waves(acc, dyn, wave, lane)) return;

    // acc[j][b][i] is out[m = 16 b + lane % 16][n = n0 + 16 j + 4 q + i]
#pragma unroll
    for (int b = 0; b < MB; b++) {
        const int64_t m = 16 * b + r;
        if (m >= p.M) continue;
#pragma unroll
        for (int j = 0; j < NB; j++) {
            const int64_t n = n0 + 16 * j + 4 * q;
            if (splits > 1) {
                __builtin_memcpy(p.part + ((int64_t)blockIdx.y * p.M + m) * p.N + n, &acc[j][b], 16);
                continue;
            }
            uint16_t o[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                float v = acc[j][b][e];
                if (p.bias) v = v + load_scalar_as_f32(p.bias, p.bias_dt, n + e);
                o[e] = bits_x<XDT>(v);
            }
            __builtin_memcpy(p.y + m * p.N + n, o, 8);
        }
    }
}

template <int XDT, int WBITS, int MB, bool HAS_OFF>
static int launch_nk_one(const WqParams& p, const WqNkPlan& pl, hipStream_t st)
{
    constexpr int NB = nk_nb(MB), COLS = 16 * NB;
    const dim3 grid((unsigned)((p.N + COLS - 1) / COLS), (unsigned)pl.splits);
    constexpr size_t lds_sum = (size_t)2 * NB * MB * 4 * 64 * 4;
    const size_t lds_tab = (size_t)pl.groups * COLS * 4;
    auto k = wq_nk_kernel<XDT, WBITS, MB, HAS_OFF>;
    static std::atomic<uint64_t> attr_set{0};   // one bit per device: the attribute belongs to the (kernel, device) pair
    if (!device_flag_test(attr_set)) {
        hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)(lds_sum > 32768 ? lds_sum : 32768));
        if (e != hipSuccess) return (int)e;
        device_flag_set(attr_set);
    }
    note_route("wq_nk", pl.splits);
    hipLaunchKernelGGL(k, grid, dim3(256), lds_sum > lds_tab ? lds_sum : lds_tab, st, p, pl.splits, pl.groups);
    if (hipError_t e = hipGetLastError(); e != hipSuccess || pl.splits == 1) return (int)e;
    launch_wq_splitk_reduce(p, pl.splits, XDT, st);
    return (int)hipGetLastError();
}
template <int XDT, int WBITS, bool HAS_OFF>
static int launch_nk_mb(const WqParams& p, const WqNkPlan& pl, hipStream_t st)
{
    if (pl.mb == 1) return launch_nk_one<XDT, WBITS, 1, HAS_OFF>(p, pl, st);
    if (pl.mb == 2) return launch_nk_one<XDT, WBITS, 2, HAS_OFF>(p, pl, st);
    return launch_nk_one<XDT, WBITS, 4, HAS_OFF>(p, pl, st);
}

// What this kernel takes with its plan, in us (median error 6 %).
static double nk_us(int wbits, bool bf16, int64_t M, int64_t N, int64_t K, const WqNkPlan& pl)
{
    const int64_t cols = 16 * nk_nb(pl.mb), kc = (pl.mb == 4 || wbits == 8) ? 64 : 128, chunks = (K + kc - 1) / kc;
    const int64_t wgs = (N + cols - 1) / cols * pl.splits, per_wave = (chunks + 4 * pl.splits - 1) / (4 * pl.splits);
    const double t = pl.mb == 4 ? 1.72 * (wbits == 8 ? 1.05 : 1.0) : (pl.mb == 2 ? 4.1 : 3.6) * (wbits == 8 ? 0.8 : 1.0);
    const double share = wgs > 256 ? (pl.mb == 4 ? 1.7 : 1.5) : 1.0;   // two workgroups on a CU
    return 6.4 + (double)per_wave * t * share * (double)((wgs + 511) / 512) * (bf16 ? 1.035 : 1.0) +
           (pl.splits > 1 ? 0.7 + 8.0 * pl.splits * (double)M * (double)N / 4.0e6 : 0.0);
}

// Does the call run here?  Looks at what both phases know: not at the weight's address, which for a FRACTAL_NZ weight is that of
// its ND copy in phase 2 alone (launch_wq_nk declines an unaligned one; the workspace has room for either outcome).
//
// Up to 16 rows the specialised kernels keep what they take (wqmm.hip): K in whole 128-element units, groups of whole chunks.
// Otherwise the estimates decide: against the streaming kernel (17 .. 32 rows, and from 33 where the many-rows kernel's shape
// conditions fail), the many-rows kernel (from 33 rows, narrow weights), and the general kernel (groups that are not whole chunks;
// fp16 with 4-bit weights, elsewhere it is never the faster one).  A short K or a wide N is theirs, a long K against a narrow N is
// cut along K here: 17 x 1024 x 11016 fp16 x int4 7.5 us there and 11.4 here, 48 x 8192 x 22896 61 and 93, but 64 x 8192 x 4104
// 50 and 25.5, 32 x 4096 x 4096 bf16 21.9 and 13.4, 64 x 4096 x 4096 23.8 and 17.5; groups of 64: 16 x 1024 x 11008 8.5 and 12.1,
// 64 x 8192 x 2048 40 and 18.  (Of 513 measured calls 492 go to the faster kernel or one within 3 % of it.)
static bool nk_wanted(const OpsnnWqmmArgs& a, WqNkPlan& pl)
{
    if ((a.w_dtype != DT_I4 && a.w_dtype != DT_I8) || (a.x_dtype != DT_F16 && a.x_dtype != DT_BF16)) return false;
    if (a.scale_dtype != a.x_dtype) return false;
    if (a.M > 64 || a.K % 32 != 0 || a.K < 256 || a.N < 256 || a.K >= (1ll << 30) || a.N >= (1ll << 30)) return false;
    if (a.w.row_stride != 1 || a.w.col_stride != a.K) return false;
    if ((uintptr_t)a.x % 16 != 0 || a.force_variant != 0) return false;
    const WqForm f = wq_form(a);
    if (f.group < a.K && f.group % 32 != 0) return false;
    if (f.stream && a.M <= 16 && a.K % 128 == 0) return false;   // (the x-in-registers kernel)
    if (!nk_plan(f.wbits, a.M, a.N, a.K, f.group, pl)) return false;
    if (f.stream && a.M <= 16) return true;
    const bool bf16 = a.x_dtype == DT_BF16;
    double other;
    if (f.stream && a.M > 32 && f.rows) {
        if (!opsnn_wq_narrow_slabs() || a.K >= 8192 || a.N > 8192) return false;   // (wide, or cut along K there)
        if (a.N > 5120 && wq_part_slices(f.wbits, a.M, a.N, a.K, f.group, true) > 1) return false;
        const int64_t kc = 4 * (128 / f.wbits), wgs = (a.N + 127) / 128;
        const double cols = wgs <= 128 && a.K % (4 * kc) == 0 ? 0.6 : (double)((wgs + 255) / 256);
        other = 6.0 + cols * (double)a.K / 4096.0 * (wq_rows_dequant_us(f.wbits, bf16) + 15.5);
    }
    else if (f.stream) {
        if (f.rows && (!opsnn_wq_narrow_slabs() || wq_part_slices(f.wbits, a.M, a.N, a.K, f.group, true) > 1)) return false;
        other = wq_stream_pass_us(f.wbits, bf16, a.M, a.N, a.K);
    }
    else if (wq_general_counts(a, f)) other = 0.94 * wq_general_pass_us(a.M, a.N, a.K);   // (in doubt the general one)
    else return true;
    return nk_us(f.wbits, bf16, a.M, a.N, a.K, pl) < other;
}
// What the kernel typically takes for a call of up to 64 rows with a shape of its own (others: a large number), for the rule of wq_wide.hip
// (488 calls, median error 4 %): us per chunk of a wave by row blocks.
double wq_nk_typical_us(const OpsnnWqmmArgs& a)
{
    static const double chunk[2][2][3] = {{{3.81, 4.21, 1.83}, {4.56, 5.01, 1.84}}, {{1.59, 2.43, 1.69}, {1.86, 2.42, 1.95}}};   // [8 bits][bf16]
    WqNkPlan pl;
    const WqForm f = wq_form(a);
    if (a.M > 64 || a.K % 32 != 0 || a.K < 256 || a.N < 256 || !nk_plan(f.wbits, a.M, a.N, a.K, f.group, pl)) return 1e30;
    const bool bf16 = a.x_dtype == DT_BF16;
    const int64_t cols = 16 * nk_nb(pl.mb), kc = (pl.mb == 4 || f.wbits == 8) ? 64 : 128, chunks = (a.K + kc - 1) / kc;
    const int64_t per_wave = (chunks + 4 * pl.splits - 1) / (4 * pl.splits);
    const double t = chunk[f.wbits == 8][bf16][pl.mb == 4 ? 2 : pl.mb - 1] + (a.offset ? (bf16 ? 0.59 : 0.12) : 0.0);
    const double cu = wq_typical_turns((a.N + cols - 1) / cols * pl.splits, 1.36) * ((double)per_wave * t + 1.24);
    return 4.5 + wq_typical_both(cu, wq_typical_mb(f.wbits, a.N, a.K) / 4.06) +
           (pl.splits > 1 ? 2.86e-6 * (double)pl.splits * (double)a.M * (double)a.N * (a.N % 4 ? 2.0 : 1.0) : 0.0);
}
// ... and if so, the workspace it needs.
bool wq_nk_wanted(const OpsnnWqmmArgs& a, uint64_t* workspace)
{
    WqNkPlan pl;
    if (!nk_wanted(a, pl)) return false;
    *workspace = pl.splits > 1 ? ((uint64_t)pl.splits * (uint64_t)a.M * (uint64_t)a.N * 4 + 255) / 256 * 256 : 0;
    return true;
}
int launch_wq_nk(const OpsnnWqmmArgs& a, hipStream_t st)
{
    WqNkPlan pl;
    if ((uintptr_t)a.w.ptr % 16 != 0 || !nk_wanted(a, pl) || (pl.splits > 1 && !a.workspace)) return OPSNN_NOT_TAKEN;
    const int wbits = a.w_dtype == DT_I4 ? 4 : 8;
    WqParams p{};
    p.group = a.group > 0 && a.group < a.K ? a.group : a.K;
    p.x = (const uint16_t*)a.x;
    p.w = (const uint8_t*)a.w.ptr; p.ldw = a.w.col_stride * wbits / 8;
    p.scale = (const uint16_t*)a.scale.ptr; p.offset = (const uint16_t*)a.offset;
    p.s_rs = a.scale.row_stride; p.s_cs = a.scale_n == 1 ? 0 : a.scale.col_stride;
    p.bias = a.bias; p.bias_dt = a.bias_dtype;
    p.y = (uint16_t*)a.y; p.M = a.M; p.N = a.N; p.K = a.K;
    p.group_shift = p.group >= p.K ? 31 : (p.group & (p.group - 1)) == 0 ? __builtin_ctzll((unsigned long long)p.group) : -1;
    p.part = (float*)a.workspace;
    if (a.x_dtype == DT_F16) {
        if (wbits == 4) return a.offset ? launch_nk_mb<DT_F16, 4, true>(p, pl, st) : launch_nk_mb<DT_F16, 4, false>(p, pl, st);
        return a.offset ? launch_nk_mb<DT_F16, 8, true>(p, pl, st) : launch_nk_mb<DT_F16, 8, false>(p, pl, st);
    }
    if (wbits == 4) return a.offset ? launch_nk_mb<DT_BF16, 4, true>(p, pl, st) : launch_nk_mb<DT_BF16, 4, false>(p, pl, st);
    return a.offset ? launch_nk_mb<DT_BF16, 8, true>(p, pl, st) : launch_nk_mb<DT_BF16, 8, false>(p, pl, st);
}

}  // namespace opsnn
