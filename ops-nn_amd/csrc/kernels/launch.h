// Internal: kernel-variant ids shared by the launchers and the selector.
#pragma once
#include "opsnn_kernels.h"

#define OPSNN_NOT_TAKEN 0x7fff0001

enum {
    OPSNN_VARIANT_AUTO = 0,
    OPSNN_VARIANT_PLAIN = 1,      // strided one-thread-per-output kernels (any shape)
    OPSNN_VARIANT_I8_256 = 2,     // int8 MFMA, 256x256 tile
    OPSNN_VARIANT_I8_128 = 3,     // int8 MFMA, 128x128 tile
    OPSNN_VARIANT_I8_256x128_S3 = 4,  // int8 MFMA, 256x128 tile, BK 64, 3 stages, 2 workgroups per CU
    OPSNN_VARIANT_I8_256_W8 = 5,  // int8 MFMA, 256x256 tile, 8 waves, BK 64, 4 stages
    OPSNN_VARIANT_I8_256_S4 = 6,  // int8 MFMA, 256x256 tile, 4 waves, BK 64, 4 stages
    OPSNN_VARIANT_I8_256_W8_K128 = 7,  // int8 MFMA, 256x256 tile, 8 waves, BK 128, 2 stages
    OPSNN_VARIANT_I8_WIDE8 = 8,   // int8 MFMA, 4 waves with 128 x 16n sub-tiles, 256 x 32n tile, n = 8..11 (ids 8..11)
    OPSNN_VARIANT_I8_WIDE11 = 11,
    OPSNN_VARIANT_I8_T32 = 12,    // int8 MFMA, the tiles of tile_plan: 32x64, 6 stages
    OPSNN_VARIANT_I8_T64 = 13,    // 64x64, 5 stages
    OPSNN_VARIANT_I8_T128 = 14,   // 128x128, 4 stages
    OPSNN_VARIANT_I8_T128x256 = 15,  // 128x256, 3 stages
    OPSNN_VARIANT_MX_128 = 16,    // MX MFMA, 128x128 tile
    OPSNN_VARIANT_MX_FP8_MFMA = 17,  // MXFP8 on the MFMA path (reduced accumulation precision, see qmm_mx.hip)
    OPSNN_VARIANT_I8_T192 = 18,   // int8 MFMA, 192x256, 2 stages
    OPSNN_VARIANT_FP8X_256x128 = 32,   // the tiles of the exact fp8 kernel (qmm_fp8_exact.hip)
    OPSNN_VARIANT_FP8X_128x256 = 33,
    OPSNN_VARIANT_FP8X_128x128 = 34,
    OPSNN_VARIANT_FP8X_192x128 = 35,
    OPSNN_VARIANT_FP8X_64x256 = 36,
};

#ifdef __cplusplus
#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#include <atomic>
namespace opsnn {
// hipFuncSetAttribute belongs to a (kernel, device) pair: launchers keep one of these masks per kernel instantiation,
// a bit per device ordinal (mod 64).  Two threads that both find the bit clear both set the attribute: harmless.
inline bool device_flag_test(const std::atomic<uint64_t>& mask)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return false;
    return (mask.load(std::memory_order_acquire) >> (dev & 63)) & 1u;
}
inline void device_flag_set(std::atomic<uint64_t>& mask)
{
    int dev = 0;
    if (hipGetDevice(&dev) == hipSuccess) mask.fetch_or(1ull << (dev & 63), std::memory_order_release);
}
}  // namespace opsnn
#endif
namespace opsnn {
// K split over workgroups for tile-kernel calls whose tiles would leave most of the chip idle (few rows against a narrow N):
// `splits` workgroups per tile each take a contiguous range of K tiles and leave fp32 partial sums in `part`
// ([splits][batch][M][N], at the front of the call's workspace); a second kernel adds them in split order, adds the bias
// and rounds.  splits <= 1: one workgroup per tile, no partial sums.
// The kernel that this thread launched last, a literal, and its K segments (opsnnDebugLastRoute).
void note_route(const char* kernel, int splits = 1);   // dispatch.hip
struct SplitK {
    int splits = 1;
    float* part = nullptr;
};
// How much of a weight that a call reads once leaves its lines in the last-level cache (256 MB): one in so many of its copies, the others go past it.
// A step works through three such weights and more, of which none is found there again when all of them pass through; past it they come faster,
// but then a weight that is used again at once is not found either.  A share of each fits for several weights in turn, and what is found and what
// comes from memory arrive side by side.  fp8_wide_kernel, us, all kept / none / every second / every fourth copy:
//                                        one weight again and again      three in turn                   1.4 GB in turn
//   132 MB, 64 x 18432 x 7168 block      34.9 / 35.9 / 33.6 / 33.9       36.2 / 36.3 / 33.7 / 34.0       36.3 / 36.3 / 35.9 / 35.5
//   132 MB, 64 x 7168 x 18432 row/column 33.4 / 38.7 / 34.4 / 35.4       37.5 / 39.2 / 34.6 / 35.3       37.5 / 39.2 / 37.1 / 36.8
//   132 MB, 20 x 18432 x 7168 MX         27.9 / 33.6 / 31.8 / 32.9       35.6 / 34.3 / 32.4 / 32.9       35.6 / 34.5 / 35.4 / 34.7
//   176 MB, 17 x 8192 x 21504 row/column 30.7 / 37.6 / 32.2 / 33.6       43.0 / 38.9 / 32.7 / 33.7       42.6 / 38.9 / 40.1 / 39.5
//   235 MB, 64 x 8192 x 28672 block      47.1 / 54.3 / 49.6 / 50.9       56.5 / 53.7 / 55.2 / 50.8       57.8 / 54.3 / 56.7 / 55.3
//   302 MB, 64 x 16384 x 18432 row/col.  73.3 / 75.7 / 61.0 / 64.7       81.0 / 74.7 / 73.8 / 66.0       80.5 / 74.4 / 73.6 / 71.2
// So every second one to 150 MB, every fourth one beyond (three such shares are the cache's size), and all of it below 100 MB, where three weights
// nearly fit as they are (88 MB, copies alone, 14.2 kept and 23.4 past it).  From two weights in turn on nothing is slower than with all of it kept;
// one weight again and again is, by 0 to 14 % (by 2 to 24 % with none kept).  Not for pieces of 64 bytes, half a line that is then fetched twice:
// 117 MB 25.0 / 27.5.
inline int weight_kept_share(int64_t bytes) { return bytes <= 100000000 ? 1 : bytes <= 150000000 ? 2 : 4; }
// How many ways a call with `tiles` output tiles, `ktiles` K tiles of `tile_us` microseconds each and `out_elems` outputs
// is split: at most one workgroup per CU, at least four K tiles per workgroup, at most sixteen ways -- and among those the
// count with the largest estimated gain, if that is at least 3 us: the loop time saved, ktiles * tile_us * (1 - 1/s), less
// a second launch (4 us) and the partial sums written and read back (2 s out_elems 4 bytes at `bytes_per_us`: fitted to
// measurements, 5e6 for the kernels that store 64-byte row pieces from 16 x 16 fragments, 2.4e6 for the 32 x 32-fragment
// kernel's 32-byte pieces).  (Measured without the traffic term: MXFP4 1024 x 4096 x 4096 in four splits 28 -> 65 us.)
inline int splitk_factor(int64_t tiles, int64_t ktiles, double tile_us, int64_t out_elems, double bytes_per_us)
{
    if (tiles <= 0 || tiles > 128) return 1;
    int64_t smax = 256 / tiles;
    if (smax > ktiles / 4) smax = ktiles / 4;
    if (smax > 16) smax = 16;
    int best = 1;
    double best_gain = 3.0;
    for (int64_t s = 2; s <= smax; s++) {
        const double gain = (double)ktiles * tile_us * (1.0 - 1.0 / (double)s) - 4.0 - 2.0 * (double)s * (double)out_elems * 4.0 / bytes_per_us;
        if (gain > best_gain) { best = (int)s; best_gain = gain; }
    }
    return best;
}
// MXFP4 on the tile kernels: 128 x 128 or 256 x 256 tiles, how many K segments, and the time in us that the choice rests on.
// Fitted to 1210 timed launches of 350 calls (M 17 .. 4096, K 1024 .. 18432 with and without a tail, N 1024 .. 28672, 1 to 4 batches), each
// as the geometric mean of its time with the weight from memory and from the last-level cache: a start, K steps of 256 elements for as
// many workgroups as a CU takes one after the other -- two small ones side by side --, the operands' bytes, the second kernel of a K split, and
// for a K that is no whole 128 the padded copies, which small tiles and segments run on and large tiles in one piece do not (median error
// 4 % on small tiles, 8 on large ones).  The launcher asks with the same sizes: what is planned cut is launched cut.
// (Planned in segments but launched in one, 594 x 16320 x 5312 took 127 us, 2456 x 10816 x 1211 105; 83 and 73 now.)
struct Mxfp4Plan {
    bool small;
    int splits;
    double us;
};
inline double mxfp4_tiles_us(bool small, int64_t M, int64_t N, int64_t K, int64_t batch, int splits)
{
    static const struct { double start, step, round, two, reduce, reduce_mb, copy, copy_mb, mb; } cost[3] = {   // mb: us per 10^6 bytes
        {3.25, 0.81, 0.0, 1.95, 2.5, 2.9, 8.5, 0.19, 0.072},    // small, up to 128 rows
        {2.8, 1.05, 0.0, 1.9, 2.6, 2.2, 9.6, 0.14, 0.114},      // small
        {3.75, 1.67, 6.5, 1.0, 3.2, 1.5, 8.3, 0.12, 0.15}};     // large
    const auto& c = cost[small ? (M <= 128 ? 0 : 1) : 2];
    const int64_t bm = small ? 128 : 256, wgs = ((M + bm - 1) / bm) * ((N + bm - 1) / bm) * batch * splits;
    const int64_t steps = ((K + 255) / 256 + splits - 1) / splits;
    double turns = (double)((wgs + 255) / 256);
    if (small && wgs > 256) turns = wgs <= 512 ? c.two : c.two * 0.5 * ((double)wgs / 512.0 + (double)((wgs + 511) / 512));
    const double mb = (double)(M + N) * (double)K * (double)batch * 0.5e-6, out = (double)M * (double)N * (double)batch * 1e-6;
    return c.start + turns * ((double)steps * c.step + c.round) + mb * c.mb + (splits > 1 ? c.reduce + c.reduce_mb * splits * out : 0.0) +
           (K % 128 && (small || splits > 1) ? c.copy + 2.0 * mb * c.copy_mb : 0.0);
}
inline Mxfp4Plan mxfp4_tile_plan(int64_t M, int64_t N, int64_t K, int64_t batch, bool may_split)
{
    Mxfp4Plan best{true, 1, 1e30};
    if (M > 128 && N > 128 && K % 128 == 0) {
        // Whole K tiles: small ones where large ones would be at most 64, a quarter of the CUs, unless the large ones in segments are
        // ahead, at 1.4 and 2.3 us a K tile (505 x 17536 x 6208 108 us on small tiles; 1024 x 4096 x 4096 22.9 against 28.0 on large ones, at 128
        // large tiles it is 42 against 32).  The estimate above chooses no better here: of 55 calls 6 became faster, 5 slower.
        const int64_t ktiles = (K + 255) / 256, out = M * N * batch;
        auto plan = [&](int64_t bm, double t, int& splits) {
            const int64_t tiles = ((M + bm - 1) / bm) * ((N + bm - 1) / bm) * batch;
            splits = may_split ? splitk_factor(tiles, ktiles, t, out, 4.0e6) : 1;
            return (double)((tiles * splits + 255) / 256) * (double)((ktiles + splits - 1) / splits) * t + (splits > 1 ? 4.0 + 8.0 * splits * (double)out / 4.0e6 : 0.0);
        };
        int s128, s256;
        const double us128 = plan(128, 1.4, s128), us256 = plan(256, 2.3, s256);
        best.small = ((M + 255) / 256) * ((N + 255) / 256) * batch <= 64 && us128 < 1.05 * us256;
        best.splits = best.small ? s128 : s256;
        best.us = mxfp4_tiles_us(best.small, M, N, K, batch, best.splits);
        return best;
    }
    for (int small = 1; small >= (M <= 128 || N <= 128 ? 1 : 0); small--) {
        const int64_t bm = small ? 128 : 256, tiles = ((M + bm - 1) / bm) * ((N + bm - 1) / bm) * batch;
        for (int s : {1, 2, 3, 4, 5, 6, 8, 12, 16}) {
            if (s > 1 && (!may_split || (K + 255) / 256 < 4 * s || tiles * s > 256)) break;
            const double us = mxfp4_tiles_us(small != 0, M, N, K, batch, s) * (s > 1 ? 1.03 : 1.0);   // (in doubt in one piece)
            if (us < best.us) best = {small != 0, s, us};
        }
    }
    return best;
}
// How a product of two K-contiguous operands whose 256 x 256 tiles would not fill the chip once (or of up to 128 rows or columns)
// is tiled (qmm_int8.hip; int8, and the 16-bit operands of gemm16.hip).  KB: bytes of K.  variant: the OPSNN_VARIANT_I8_*
// tile, 0 if the shape is outside; splits: K segments; us: the estimate that the choice rests on.
struct TilePlan {
    int variant, splits;
    double us;
};
TilePlan tile_plan(int64_t M, int64_t N, int64_t KB, int64_t batch, bool may_split, bool tiles_of_32 = true);

// The tile (OPSNN_VARIANT_FP8X_*) and the K segments of a call on the exact fp8 kernel (qmm_fp8_exact.hip).
struct Fp8xPlan {
    int tile, splits;
    double us;   // the estimate that the choice rests on
};
enum Fp8xForm { FP8X_BLOCK, FP8X_PLAIN, FP8X_MX };   // block scales, row / column scales, MX scales
Fp8xPlan fp8x_plan(int64_t M, int64_t N, int64_t K, int64_t batch, Fp8xForm form, bool may_split);

// Whether a call of fp8 operands with few rows runs on the stream kernel of qmm_fp8_stream.hip, and how: row and column blocks of 16 per
// workgroup, K segments (sizes, types and strides only: both phases of a call ask).
struct Fp8StreamPlan {
    int mb, nb, splits;
    bool wide;   // the waves share x1 and each K tile, or each has a quarter of K
};
bool fp8_stream_plan(const OpsnnQmmArgs& a, Fp8xForm form, bool may_split, Fp8StreamPlan& pl);

// How the x-in-registers kernel (weight-only, up to 16 rows of x) covers K.  A workgroup holds `nw` waves x `nch` chunks
// (of 64 weight bytes): 16 x 4, 8-bit weights also 16 x 8, or 8 x 4 / 8 x 8.  A K that is exactly one such shape runs on
// one workgroup per row block range; any other K of whole 128-element units goes in `splits` segments of 16 x 4 chunks
// (else of 8 x 4), one workgroup column per segment, the last one with idle chunks past the end of K (`exact` false) when
// that wastes at most a fifth of K's chunks; with more than one segment the columns leave fp32 partial sums
// [splits][M][N] at the front of the workspace.  False: the kernel does not take this K.
struct WqXregPlan {
    int nw, nch, splits;
    bool exact;
};
inline bool wq_xreg_plan(int wbits, int64_t M, int64_t K, WqXregPlan& pl)
{
    const int64_t kc = 4 * (128 / wbits);
    if (M < 1 || M > 16 || K < 128 || K % 128 != 0) return false;
    const int64_t nch = K / kc;
    if (nch == 64) { pl = {16, 4, 1, true}; return true; }
    if (wbits == 8 && nch == 128) { pl = {16, 8, 1, true}; return true; }
    if (nch == 32) { pl = {8, 4, 1, true}; return true; }
    const int64_t s64 = (nch + 63) / 64, w64 = s64 * 64 - nch, s32 = (nch + 31) / 32, w32 = s32 * 32 - nch;
    if (s64 == 1 && w64 * 5 <= nch) { pl = {16, 4, 1, false}; return true; }   // one workgroup, its last waves idle
    if (s32 <= 16 && w32 * 5 <= nch) { pl = {8, 4, (int)s32, w32 == 0}; return true; }
    if (s64 <= 16 && w64 * 5 <= nch) { pl = {16, 4, (int)s64, w64 == 0}; return true; }
    return false;
}
// the count of partial-sum slices that plan needs (0: none)
inline int wq_xreg_splits(int wbits, int64_t M, int64_t K)
{
    WqXregPlan pl;
    return (wq_xreg_plan(wbits, M, K, pl) && pl.splits > 1) ? pl.splits : 1;
}
// Row slabs of the many-rows weight-only kernel for a narrow N.  Its workgroups take 128 columns each, so one pass over a
// narrow weight leaves most CUs idle, and passes launched one after the other do not overlap (4096 x 4096 int4: 32
// workgroups, 256 rows 56 us, 1024 rows in four passes 219 us).  With at most 128 workgroups per pass and more than 64
// rows the rows are cut into equal slabs of 64 .. 256 rows, as many as give every CU a workgroup in one round, and all
// slabs go out in one launch (grid.y).  Returns the slab's rows, or 0 where the one-pass-at-a-time order stays.
inline int64_t wq_narrow_slab_rows(int64_t M, int64_t N, bool on)
{
    const int64_t wgs = (N + 127) / 128;
    if (M <= 64 || wgs > 128 || !on) return 0;
    int64_t n = 256 / wgs;
    if (n > (M + 63) / 64) n = (M + 63) / 64;
    if (n < (M + 255) / 256) n = (M + 255) / 256;
    if (n < 2) return 0;
    return ((M + n - 1) / n + 15) / 16 * 16;
}
// The same kernel, from 17 rows: a narrow N leaves CUs without a workgroup even with all row slabs in one
// launch (64 rows against 28672 x 8192: 64 workgroups of 128 columns), and a long K makes each of them slow.  Then K is
// cut into segments, one per blockIdx.z, whose fp32 partial sums a second kernel adds in segment order.  Segments are
// whole units (a slab of x of the 64-row instance -- two chunks of 128 bytes of a weight row -- or a group where that is
// longer), as equal as that allows, at least 2048 k each.  Returns the segment count (1: no split) and the unit.
// (Measured, int4 with groups of 128, 64 rows: 14336 x 4096 64 -> 22 us, 28672 x 8192 124 -> 66, 8192 x 8192 30 -> 24; a K
// of 4096 lost 2 to 6 us to the second kernel, and so did two segments of 128 workgroups at K = 8192; 64 x 7168 x 7168, where
// the 64-column workgroups cannot run, 42 -> 26.)
inline int wq_rows_ksplit(int wbits, int64_t M, int64_t N, int64_t K, int64_t group, bool on, int64_t* kunit = nullptr)
{
    if (!on || M < 17 || N % 32 != 0 || N < 256 || K < 4096 || K >= (1ll << 23)) return 1;
    const int64_t slab = wq_narrow_slab_rows(M, N, on);
    if (M > 64 && slab == 0) return 1;
    const int64_t slabs = slab ? (M + slab - 1) / slab : 1;
    const int64_t wgs = slabs * ((N + 127) / 128), kx = 2 * 4 * (128 / wbits);
    int64_t unit = kx;
    if (group < K) {
        if (group > kx) unit = group;
        if (unit % group != 0 || unit % kx != 0) return 1;
    }
    if (wgs > 128 || K % unit != 0) return 1;
    // (below 8192 only where the 64-column workgroups, which double the workgroups without a second kernel, cannot run: they
    // want K in whole slabs of four chunks; and from 33 rows: 17 x 5120 x 5120 int4 took 19 us on the streaming kernel, 22 here)
    if (K < 8192 && (K % (2 * kx) == 0 || wgs > 64 || M < 33)) return 1;
    int64_t s = 256 / wgs;
    if (s > 8) s = 8;
    if (s > K / 2048) s = K / 2048;
    if (s > K / unit) s = K / unit;
    if (s == 2 && wgs > 64 && K < 12288) return 1;
    if (kunit) *kunit = unit;
    return s < 2 ? 1 : (int)s;
}
// fp32 partial-sum slices [slices][M][N] at the front of a weight-only call's workspace (1: none)
inline int wq_part_slices(int wbits, int64_t M, int64_t N, int64_t K, int64_t group, bool narrow_on)
{
    if (M <= 16) return wq_xreg_splits(wbits, M, K);
    return wq_rows_ksplit(wbits, M, N, K, group, narrow_on);
}
// The fp8 / int8 decode kernel (qmm_fp8_decode.hip, up to 16 rows of x1): K in blocks of 128 that the NW = 16 or 8 waves
// of a workgroup share, NBLK each (a wave keeps its blocks of x1 in registers: 16 waves up to 4, not 3; 8 waves up to 7).
// A K that the waves of one workgroup share exactly runs as one segment; any other whole number of blocks in 1 .. 16
// segments of NW * NBLK blocks, the last one with idle waves (K a whole number of NBLK blocks): the layout with the fewest
// wave slots, then the fewest segments.  More than one segment needs room for fp32 partial sums (may_split).
// (w4: the fp8 x fp4 MX form of the kernel, which has no instance of 16 waves with one block each.)
struct QmmDecodePlan { int nw = 0, nblk = 0, splits = 1; };
inline bool qmm_decode_plan(int64_t K, bool may_split, QmmDecodePlan& pl, bool w4 = false)
{
    if (K <= 0 || K % 128 != 0) return false;
    const int64_t nb = K / 128;
    if (nb % 16 == 0 && nb / 16 <= 4 && nb / 16 != 3 && !(w4 && nb == 16)) { pl.nw = 16; pl.nblk = (int)(nb / 16); pl.splits = 1; return true; }
    if (nb % 8 == 0 && nb / 8 <= 7) { pl.nw = 8; pl.nblk = (int)(nb / 8); pl.splits = 1; return true; }
    static const int shapes[10][2] = {{16, 4}, {16, 2}, {16, 1}, {8, 7}, {8, 6}, {8, 5}, {8, 4}, {8, 3}, {8, 2}, {8, 1}};
    int64_t best_slots = 0;
    bool found = false;
    for (const auto& sh : shapes) {
        const int nw = sh[0], nblk = sh[1];
        if (nb % nblk != 0 || (w4 && nw == 16 && nblk == 1)) continue;
        const int64_t waves = nb / nblk, s = (waves + nw - 1) / nw;
        if (s > 16 || (s > 1 && !may_split)) continue;
        const int64_t slots = s * nw * nblk;
        if (!found || slots < best_slots || (slots == best_slots && s < pl.splits)) {
            found = true; best_slots = slots; pl.nw = nw; pl.nblk = nblk; pl.splits = (int)s;
        }
    }
    return found;
}
// Opened by every exported matmul entry point for the time it enqueues its launches (weight_cache.hip): copies that the
// weight cache hands out inside the scope cannot be evicted before it closes; bypass = true switches the cache off for
// this thread while the scope is open.  Scopes nest; the pins drop when the outermost one closes.
class WeightCacheScope {
public:
    explicit WeightCacheScope(bool bypass = false);
    ~WeightCacheScope();
    WeightCacheScope(const WeightCacheScope&) = delete;
    WeightCacheScope& operator=(const WeightCacheScope&) = delete;
private:
    bool saved_bypass_;
};
}  // namespace opsnn
#endif
