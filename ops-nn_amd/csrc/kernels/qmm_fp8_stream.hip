// fp8 e4m3 x fp8 e4m3 with few rows of x1 (block scales; row and column scales; MX scales): exact products as in qmm_fp8_exact.hip,
// organised as a stream over x2.
//
//   block scales    out[m,n] = cast( sum_kb ( sum_{k in block kb} x1[m,k] x2[k,n] ) * ( s1[m/gsM, kb] * s2[kb, n/128] ) )
//   row / column    out[m,n] = cast( (sum_k x1[m,k] x2[k,n]) * cs[n] * rs[m] + bias[n] )
//   MX              out[m,n] = cast( sum_k (x1[m,k] 2^(a[m,k/32]-127)) * (x2[k,n] 2^(b[n,k/32]-127)) + bias[n] )
//
// Formulas: matmul/quant_batch_matmul_v3/tests/assets/qbmmv3_kernel_golden.py:153-234, :237-387.
//
// What bounds such a call, x2's stream from memory apart, is the memory pipeline of a CU: a load whose neighbouring lanes lie in
// different rows -- the operand layout of the matrix instructions, 16 rows per 16 lanes -- takes 66 clocks per KB, one lane after the
// other; the same KB with four neighbouring lanes in one 64-byte row piece takes 33 (measured, L2 resident).  So both operands travel
// global -> LDS in that order, 16 bytes per lane, fp8 as they are: half the bytes that x1 widened to 16 bits by a launch of its own
// would be, and no such launch.  From LDS the fragments come in the matrix layout, conflict-free.
//
// The four waves of a workgroup (one per SIMD) share nothing until the end: each owns a quarter of the workgroup's K and all of its
// 16 MB x 16 NB outputs, with a ring of S K tiles of 64 of its own.  It waits for its own copies by count; there is no barrier in the
// loop.  The four sums meet in LDS in wave order; blockIdx.y cuts K further, with fp32 partial sums for fp8_stream_reduce_kernel.
// (What it measured, before and now, x2 from memory, a call: row / column scales 64 x 4096 x 4096 33.2 -> 13.0 us, block scales
// 24 x 2560 x 1536 19.8 -> 7.0, 64 x 18432 x 7168 50.2 -> 40.3 -- 3.3 TB/s, of 5.6 that the copies alone reach --, 32 x 7296 x 22529 92 -> 40,
// MX 64 x 10496 x 1152 25.0 -> 14.3.)
// An operand piece of 16 bytes is two k steps of v_mfma_f32_16x16x32_{f16,bf16}, cut the same way for x1 and x2.
#include <cmath>

#include "launch.h"
#include "common.hip.h"

namespace opsnn {
namespace {

struct Fp8StreamParams {
    const uint8_t *a, *b;         // x1 [M, K], x2 as [N, K]
    int64_t lda, ldb;
    void* out; int out_dt;
    int M, N, tiles;              // tiles of 64 along K
    int splits;
    const float* s1; int64_t s1_rs, s1_cs;   // block scales
    const float* s2; int64_t s2_rs, s2_cs;
    int gsM;
    const uint8_t *sa, *sb;       // MX scales, [rows, K / 32] bytes
    int64_t sa_rs, sb_rs;
    const float *rs, *cs;         // row / column scales, strides 0 (one scale) or 1
    int rs_stride, cs_stride;
    const float* bias;
    float* part;                  // [splits][M][N]
    int kept;                     // one in so many of x2's copies leaves its lines in the last-level cache
};

template <int FORM>
__device__ __forceinline__ v4i widen8(uint32_t d0, uint32_t d1, float sc)
{
    if constexpr (FORM == FP8X_MX) {
        typedef __bf16 b2v __attribute__((ext_vector_type(2)));
        const b2v w0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(d0, sc, false), w1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(d0, sc, true);
        const b2v w2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(d1, sc, false), w3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(d1, sc, true);
        return (v4i){(int)__builtin_bit_cast(uint32_t, w0), (int)__builtin_bit_cast(uint32_t, w1), (int)__builtin_bit_cast(uint32_t, w2), (int)__builtin_bit_cast(uint32_t, w3)};
    } else {
        typedef _Float16 h2v __attribute__((ext_vector_type(2)));
        const h2v w0 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(d0, 1.0f, false), w1 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(d0, 1.0f, true);
        const h2v w2 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(d1, 1.0f, false), w3 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(d1, 1.0f, true);
        return (v4i){(int)__builtin_bit_cast(uint32_t, w0), (int)__builtin_bit_cast(uint32_t, w1), (int)__builtin_bit_cast(uint32_t, w2), (int)__builtin_bit_cast(uint32_t, w3)};
    }
}
// Asynchronous copies of one dword, or of 16 bits into a dword, per lane, by the first LANES lanes (copy4_sbase's conditions).  Every
// lane is a request of its own here, so that only as many take part as there are rows.
template <int LANES>
__device__ __forceinline__ void copy4_lanes(const void* base, uint32_t voff, uint32_t lds)
{
    uint64_t all;
    asm volatile("s_mov_b64 %0, exec\n\ts_mov_b64 exec, %4\n\ts_mov_b32 m0, %1\n\ts_nop 4\n\tglobal_load_lds_dword %2, %3\n\ts_mov_b64 exec, %0"
                 : "=&s"(all) : "s"(lds), "v"(voff), "s"(base), "s"(LANES >= 64 ? ~0ull : (1ull << (LANES & 63)) - 1) : "memory", "m0");
}
template <int LANES>
__device__ __forceinline__ void copy2_lanes(const void* base, uint32_t voff, uint32_t lds)
{
    uint64_t all;
    asm volatile("s_mov_b64 %0, exec\n\ts_mov_b64 exec, %4\n\ts_mov_b32 m0, %1\n\ts_nop 4\n\tglobal_load_lds_ushort %2, %3\n\ts_mov_b64 exec, %0"
                 : "=&s"(all) : "s"(lds), "v"(voff), "s"(base), "s"(LANES >= 64 ? ~0ull : (1ull << (LANES & 63)) - 1) : "memory", "m0");
}

// bytes of a K tile in a wave's ring, copies per tile
template <int MB, int NB, int FORM> constexpr int fs_tile = (MB + NB) * 1024 + (FORM == FP8X_BLOCK ? 256 : FORM == FP8X_MX ? 256 + (NB + 3) / 4 * 256 : 0);
template <int MB, int NB, int FORM> constexpr int fs_copies = MB + NB + (FORM == FP8X_BLOCK ? 1 : FORM == FP8X_MX ? 1 + (NB + 3) / 4 : 0);
// stages: what the 160 KB of a CU hold, 8 at most
template <int FORM> constexpr int fs_table = FORM == FP8X_BLOCK ? 4096 : 0;   // x2's block scales: 256 per wave
constexpr int at_most_8(int v) { return v > 8 ? 8 : v; }
template <int MB, int NB, int FORM> constexpr int fs_stages = at_most_8((163840 - fs_table<FORM>) / 4 / fs_tile<MB, NB, FORM>);

// what the kernels add behind the sums, 4 columns of row m from n on (n < N)
template <int FORM>
__device__ __forceinline__ void fs_finish(const Fp8StreamParams& p, int m, int n, v4f& v)
{
    if constexpr (FORM == FP8X_PLAIN) {
        const float rsv = p.rs[(int64_t)m * p.rs_stride];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int ni = n + e < p.N ? n + e : p.N - 1;
            v[e] = (v[e] * p.cs[(int64_t)ni * p.cs_stride]) * rsv;
        }
    }
    if (p.bias) {
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = v[e] + p.bias[n + e < p.N ? n + e : p.N - 1];
    }
}

// x2's block scales for a wave's blocks of K and its one column block, fetched into LDS in front of the tiles.  (A scalar load per
// block is waited for with every LDS read of the tile, the two share a counter and arrive in any order; a vector load in the loop is
// waited for with every copy under way: 1300 clocks a tile, 700 so.)
constexpr int FS_MOST_BLOCKS = 256;
__device__ __forceinline__ void fetch_scale2(const Fp8StreamParams& p, int kb0, int blocks, int n, uint32_t lds)
{
    const float* const base = p.s2 + kb0 * p.s2_rs + (n / 128) * p.s2_cs;
    for (int i = 0; i < blocks; i += 64) {   // (past the end: the last one again)
        const int j = i + (int)(threadIdx.x & 63);
        copy4_lanes<64>(base, (uint32_t)((j < blocks ? j : blocks - 1) * p.s2_rs * 4), __builtin_amdgcn_readfirstlane(lds + 4 * i));
    }
}

// four columns of row m from n on: the workgroup's own segment of a K split, or the outputs
template <int FORM>
__device__ __forceinline__ void fs_store(const Fp8StreamParams& p, int m, int n, v4f sum)
{
    if (m >= p.M || n >= p.N) return;
    const bool whole = n + 3 < p.N;
    if (p.splits > 1) {
        float* dst = p.part + ((int64_t)blockIdx.y * p.M + m) * p.N + n;
        if (whole) __builtin_memcpy(dst, &sum, 16);
        else {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (n + e < p.N) dst[e] = sum[e];
        }
        return;
    }
    fs_finish<FORM>(p, m, n, sum);
    const int64_t at = (int64_t)m * p.N + n;
    if (p.out_dt == DT_F32) {
        float* dst = (float*)p.out + at;
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (n + e < p.N) dst[e] = sum[e];
    } else {
        const v4us o = p.out_dt == DT_BF16 ? pack4_b16<DT_BF16>(sum) : pack4_b16<DT_F16>(sum);
        uint16_t* dst = (uint16_t*)p.out + at;
        if (whole) __builtin_memcpy(dst, &o, 8);
        else {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (n + e < p.N) dst[e] = o[e];
        }
    }
}

template <int MB, int NB, int FORM, int S>
__global__ __launch_bounds__(256, 1) void fp8_stream_kernel(Fp8StreamParams p)
{
    constexpr int TILE = fs_tile<MB, NB, FORM>, CPT = fs_copies<MB, NB, FORM>;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, q = lane >> 4;
    const int n0 = (int)blockIdx.x * (16 * NB), m0 = (int)blockIdx.z * (16 * MB);

    // this wave's K tiles t0 .. t0 + nt - 1 (whole blocks of 128; a last half one belongs to the last)
    const int units = (p.tiles + 1) / 2;
    const int s0 = (int)((int64_t)blockIdx.y * units / p.splits), s1 = (int)((int64_t)(blockIdx.y + 1) * units / p.splits);
    const int t0 = 2 * (s0 + (s1 - s0) * wave / 4);
    int t1 = 2 * (s0 + (s1 - s0) * (wave + 1) / 4);
    if (t1 > p.tiles) t1 = p.tiles;
    const int nt = t1 - t0;

    // copies: lane l fetches piece (l % 4) ^ key of row l / 4 of a block of 16 rows to 16 l; key(row) = 2 (row / 8) makes the sixteen
    // lanes that a 16-byte LDS read serves together (lane bits 2 and 4 unequal or equal) hit sixteen different 16-byte columns
    const int crow = lane >> 2, cpiece = (lane & 3) ^ ((crow >> 3) << 1);
    uint32_t xo[MB], wo[NB], so = 0, swo[(NB + 3) / 4];
#pragma unroll
    for (int b = 0; b < MB; b++) {
        const int m = m0 + 16 * b + crow < p.M ? m0 + 16 * b + crow : p.M - 1;
        xo[b] = (uint32_t)(m * p.lda) + 16 * cpiece;
    }
#pragma unroll
    for (int j = 0; j < NB; j++) {
        const int n = n0 + 16 * j + crow < p.N ? 16 * j + crow : p.N - 1 - n0;
        wo[j] = (uint32_t)(n * p.ldb) + 16 * cpiece;
    }
    if constexpr (FORM != FP8X_PLAIN) {   // scales: one row per lane
        const int ml = lane < 16 * MB ? lane : 16 * MB - 1, m = m0 + ml < p.M ? m0 + ml : p.M - 1;
        so = FORM == FP8X_BLOCK ? (uint32_t)(m / p.gsM * p.s1_rs * 4) : (uint32_t)(m * p.sa_rs);
    }
    if constexpr (FORM == FP8X_MX) {
#pragma unroll
        for (int j = 0; j < (NB + 3) / 4; j++) {
            const int nl = 64 * j + lane < 16 * NB ? 64 * j + lane : 16 * NB - 1;
            swo[j] = (uint32_t)((n0 + nl < p.N ? nl : p.N - 1 - n0) * p.sb_rs);
        }
    }
    (void)so; (void)swo;
    const uint8_t* const wbase = p.b + (int64_t)n0 * p.ldb;
    const uint8_t* const sbase = FORM == FP8X_MX ? p.sb + (int64_t)n0 * p.sb_rs : nullptr;
    const uint32_t ring = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)smem + wave * (S * TILE);
    auto issue = [&](int t, int stage) {
        const int64_t k = (int64_t)__builtin_amdgcn_readfirstlane(t0 + (t < nt ? t : nt - 1)) * 64;   // past the end: a harmless copy once more, so that the counts hold
        const uint32_t at = __builtin_amdgcn_readfirstlane(ring + stage * TILE);
#pragma unroll
        for (int b = 0; b < MB; b++) copy16_sbase(p.a + k, xo[b], at + b * 1024);
#pragma unroll
        for (int j = 0; j < NB; j++) copy16_sbase(wbase + k, wo[j], at + (MB + j) * 1024);
        if constexpr (FORM == FP8X_BLOCK) copy4_lanes<16 * MB>((const char*)p.s1 + (k >> 7) * p.s1_cs * 4, so, at + (MB + NB) * 1024);
        if constexpr (FORM == FP8X_MX) {
            copy2_lanes<16 * MB>(p.sa + (k >> 5), so, at + (MB + NB) * 1024);
#pragma unroll
            for (int j = 0; j < (NB + 3) / 4; j++) copy2_lanes<(NB < 4 ? 16 * NB : 64)>(sbase + (k >> 5), swo[j], at + (MB + NB) * 1024 + 256 * (1 + j));
        }
    };

    v4f acc[NB][MB];
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
        for (int b = 0; b < MB; b++) acc[j][b] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};

    // a tile's fragments: 16 bytes per lane and row block (two k steps), and the scales of its rows
    struct Frags {
        v4i x[MB], w[NB];
        float xs[MB], ws[NB];
    };
    const char* const mine = smem + wave * (S * TILE);
    const int fat = r * 64 + ((q ^ ((r >> 3) << 1)) << 4);
    auto read = [&](Frags& f, int stage) {
        const char* at = mine + stage * TILE;
#pragma unroll
        for (int b = 0; b < MB; b++) f.x[b] = *(const v4i*)(at + fat + b * 1024);
#pragma unroll
        for (int j = 0; j < NB; j++) f.w[j] = *(const v4i*)(at + fat + (MB + j) * 1024);
        if constexpr (FORM == FP8X_BLOCK) {
#pragma unroll
            for (int b = 0; b < MB; b++) f.xs[b] = *(const float*)(at + (MB + NB) * 1024 + (16 * b + r) * 4);
        }
        if constexpr (FORM == FP8X_MX) {
#pragma unroll
            for (int b = 0; b < MB; b++) f.xs[b] = e8m0_to_f32(*(const uint8_t*)(at + (MB + NB) * 1024 + (16 * b + r) * 4 + (q >> 1)));
#pragma unroll
            for (int j = 0; j < NB; j++) f.ws[j] = e8m0_to_f32(*(const uint8_t*)(at + (MB + NB) * 1024 + 256 + (16 * j + r) * 4 + (q >> 1)));
        }
    };
    // sums of the current 128 elements: folded into acc with the block's scale, or just added (a chain over the wave's whole K inside the
    // matrix instruction loses more: MX 64 x 18432 x 7168 2.9e-7 of the result's norm against 1.9e-7)
    v4f part[NB][MB];
    auto multiply = [&](const Frags& f, auto closes, float s2) {   // closes: the second tile of a block of 128
#pragma unroll
        for (int h = 0; h < 2; h++) {
            v4i x[MB];
#pragma unroll
            for (int b = 0; b < MB; b++) x[b] = widen8<FORM>((uint32_t)f.x[b][2 * h], (uint32_t)f.x[b][2 * h + 1], f.xs[b]);
#pragma unroll
            for (int j = 0; j < NB; j++) {
                const v4i w = widen8<FORM>((uint32_t)f.w[j][2 * h], (uint32_t)f.w[j][2 * h + 1], f.ws[j]);
#pragma unroll
                for (int b = 0; b < MB; b++) {
                    if constexpr (FORM == FP8X_MX) part[j][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, w), __builtin_bit_cast(v8bf, x[b]), part[j][b], 0, 0, 0);
                    else part[j][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, w), __builtin_bit_cast(v8h, x[b]), part[j][b], 0, 0, 0);
                }
            }
        }
        if constexpr (decltype(closes)::value) {
#pragma unroll
            for (int b = 0; b < MB; b++) {
                const float sc = FORM == FP8X_BLOCK ? f.xs[b] * s2 : 1.0f;
#pragma unroll
                for (int j = 0; j < NB; j++)
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[j][b][e] = FORM == FP8X_BLOCK ? __builtin_fmaf(part[j][b][e], sc, acc[j][b][e]) : acc[j][b][e] + part[j][b][e];
            }
        }
    };
    auto open = [&]() {
#pragma unroll
        for (int j = 0; j < NB; j++)
#pragma unroll
            for (int b = 0; b < MB; b++) part[j][b] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
    };

    if (nt > 0) {
        // (16 NB columns from a multiple of 16 NB on: one scale block)
        if constexpr (FORM == FP8X_BLOCK) fetch_scale2(p, t0 >> 1, nt >> 1, n0, (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)smem + 4 * S * TILE + wave * (4 * FS_MOST_BLOCKS));
        // tile t + 1 is read while tile t multiplies; tile t + S goes where tile t was, whose fragments have arrived by then
#pragma unroll
        for (int i = 0; i < S; i++) issue(i, i);
        wait_copies<(S - 1) * CPT>();
        Frags f0, f1;
        read(f0, 0);
        int at = 0;
        auto next = [&](int v) { return v + 1 < S ? v + 1 : 0; };
        for (int t = 0; t < nt; t += 2) {
            wait_copies<(S - 2) * CPT>();
            issue(t + S, at); at = next(at);
            read(f1, at);
            __builtin_amdgcn_sched_barrier(0);
            float sc = 1.0f;
            if constexpr (FORM == FP8X_BLOCK) sc = *(const float*)(smem + 4 * S * TILE + wave * (4 * FS_MOST_BLOCKS) + 4 * (t >> 1));
            open();
            if (t + 1 >= nt) {   // a last half block (K % 128 == 64, not with block scales)
                multiply(f0, std::true_type{}, sc);
                break;
            }
            multiply(f0, std::false_type{}, sc);
            wait_copies<(S - 2) * CPT>();
            issue(t + 1 + S, at); at = next(at);
            read(f0, at);
            __builtin_amdgcn_sched_barrier(0);
            multiply(f1, std::true_type{}, sc);
        }
    }
    wait_copies<0>();
    __syncthreads();   // the rings make room for the sums

    // acc[j][b][e]: n = n0 + 16 j + 4 q + e, m = m0 + 16 b + r, over this wave's part of K
    float* const red = (float*)smem;
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
        for (int b = 0; b < MB; b++) *(v4f*)(red + (wave * (NB * MB) + j * MB + b) * 256 + lane * 4) = acc[j][b];
    __syncthreads();
    for (int t = tid; t < NB * MB * 64; t += 256) {
        v4f sum = *(const v4f*)(red + t * 4);
#pragma unroll
        for (int i = 1; i < 4; i++) {
            const v4f o = *(const v4f*)(red + (i * (NB * MB)) * 256 + t * 4);
#pragma unroll
            for (int e = 0; e < 4; e++) sum[e] = sum[e] + o[e];
        }
        const int j = (t >> 6) / MB, b = (t >> 6) % MB;
        const int m = m0 + 16 * b + (t & 15), n = n0 + 16 * j + 4 * ((t >> 4) & 3);
        fs_store<FORM>(p, m, n, sum);
    }
}

// ---- the same with a weight whose stream is the time: the workgroup's waves share x1's tile ----
// Four waves own 16 NB columns each and all 16 MB rows; K tiles of 128 in a ring of S stages for the workgroup, one barrier per tile.
// (With a ring per wave, x1's share of the LDS is four times as large and too few bytes of x2 are in flight: 64 x 18432 x 7168 stays at
// 2.7 TB/s.)  Rows of 128 bytes, 16-byte chunk c of row r at c ^ (r / 2 % 8).
template <int MB, int NB, int FORM> constexpr int fw_tile = MB * 2048 + NB * 8192 + (FORM == FP8X_BLOCK ? 1024 : FORM == FP8X_MX ? 1024 + 1024 : 0);
// KEPT: all of x2 by way of the last-level cache (1), or one in so many of a wave's copies of a tile and the others past it (weight_kept_share; a
// flag tested in the loop took half of the gain).
template <int MB, int NB, int FORM, int S, int KEPT>
__global__ __launch_bounds__(256, 2) void fp8_wide_kernel(Fp8StreamParams p)
{
    constexpr int TILE = fw_tile<MB, NB, FORM>;
    constexpr int XC = MB == 4 ? 2 : 1, CPT = XC + 2 * NB + (FORM == FP8X_BLOCK ? 1 : FORM == FP8X_MX ? 2 : 0);
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, q = lane >> 4;
    const int n0 = ((int)blockIdx.x * 4 + wave) * (16 * NB), m0 = (int)blockIdx.z * (16 * MB);   // this wave's first column (may lie past N)
    const int units = p.tiles / 2;
    const int t0 = (int)((int64_t)blockIdx.y * units / p.splits), nt = (int)((int64_t)(blockIdx.y + 1) * units / p.splits) - t0;

    // copies: eight rows of 128 bytes each; x1's tile is shared out over the waves (MB = 1: twice the same two), a wave's own columns its own
    const int crow = lane >> 3;
    uint32_t xo[XC], wo[2 * NB], so = 0, swo = 0;
#pragma unroll
    for (int i = 0; i < XC; i++) {
        const int row = ((wave * XC + i) * 8 + crow) % (16 * MB), m = m0 + row < p.M ? m0 + row : p.M - 1;
        xo[i] = (uint32_t)(m * p.lda) + 16 * ((lane & 7) ^ ((row >> 1) & 7));
    }
    const int nb0 = n0 < p.N ? n0 : p.N - 1;   // (base of this wave's columns; past N everything repeats the last one)
#pragma unroll
    for (int i = 0; i < 2 * NB; i++) {
        const int row = i * 8 + crow, n = n0 + row < p.N ? n0 + row : p.N - 1;
        wo[i] = (uint32_t)((n - nb0) * p.ldb) + 16 * ((lane & 7) ^ ((row >> 1) & 7));
    }
    const int srow = wave * 4 * MB + (lane < 4 * MB ? lane : 4 * MB - 1);   // scales: a quarter of x1's rows per wave
    if constexpr (FORM != FP8X_PLAIN) {
        const int m = m0 + srow < p.M ? m0 + srow : p.M - 1;
        so = FORM == FP8X_BLOCK ? (uint32_t)(m / p.gsM * p.s1_rs * 4) : (uint32_t)(m * p.sa_rs);
    }
    if constexpr (FORM == FP8X_MX) {
        const int row = lane < 16 * NB ? lane : 16 * NB - 1, n = n0 + row < p.N ? n0 + row : p.N - 1;
        swo = (uint32_t)((n - nb0) * p.sb_rs);
    }
    (void)so; (void)swo;
    const uint8_t* const wbase = p.b + (int64_t)nb0 * p.ldb;
    const uint8_t* const sbase = FORM == FP8X_MX ? p.sb + (int64_t)nb0 * p.sb_rs : nullptr;
    const uint32_t ring = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)smem;
    auto issue = [&](int t, int stage) {
        const int64_t k = (int64_t)__builtin_amdgcn_readfirstlane(t0 + (t < nt ? t : nt - 1)) * 128;
        const uint32_t at = __builtin_amdgcn_readfirstlane(ring + stage * TILE);
#pragma unroll
        for (int i = 0; i < XC; i++) copy16_sbase(p.a + k, xo[i], at + ((wave * XC + i) * 1024) % (MB * 2048));
#pragma unroll
        for (int i = 0; i < 2 * NB; i++) {
            if (i % KEPT != 0) copy16_sbase_once(wbase + k, wo[i], at + MB * 2048 + (wave * 2 * NB + i) * 1024);
            else copy16_sbase(wbase + k, wo[i], at + MB * 2048 + (wave * 2 * NB + i) * 1024);
        }
        const uint32_t sc = at + MB * 2048 + NB * 8192 + wave * 256;
        if constexpr (FORM == FP8X_BLOCK) copy4_lanes<4 * MB>((const char*)p.s1 + (k >> 7) * p.s1_cs * 4, so, sc);
        if constexpr (FORM == FP8X_MX) {
            copy4_lanes<4 * MB>(p.sa + (k >> 5), so, sc);
            copy4_lanes<16 * NB>(sbase + (k >> 5), swo, sc + 1024);
        }
    };

    v4f acc[NB][MB];
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
        for (int b = 0; b < MB; b++) acc[j][b] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
    const int key = (r >> 1) & 7;
    struct Frags {   // a tile's fragments: 2 x 16 bytes per lane and row block (four k steps), and the scales of its rows
        v4i x[2][MB], w[2][NB];
        float xs[1][MB], ws[1][NB];   // (MX: the four scale bytes of the row)
    };
    auto read = [&](Frags& f, int stage) {
        const char* const at = smem + stage * TILE;
        const char* const sc = at + MB * 2048 + NB * 8192;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int c = ((4 * h + q) ^ key) * 16;
#pragma unroll
            for (int b = 0; b < MB; b++) f.x[h][b] = *(const v4i*)(at + (16 * b + r) * 128 + c);
#pragma unroll
            for (int j = 0; j < NB; j++) f.w[h][j] = *(const v4i*)(at + MB * 2048 + (wave * 16 * NB + 16 * j + r) * 128 + c);
        }
        if constexpr (FORM == FP8X_BLOCK) {
#pragma unroll
            for (int b = 0; b < MB; b++) { const int row = 16 * b + r; f.xs[0][b] = *(const float*)(sc + row / (4 * MB) * 256 + row % (4 * MB) * 4); }
        }
        if constexpr (FORM == FP8X_MX) {   // piece q of half h lies in block 2 h + q / 2
#pragma unroll
            for (int b = 0; b < MB; b++) { const int row = 16 * b + r; f.xs[0][b] = *(const float*)(sc + row / (4 * MB) * 256 + row % (4 * MB) * 4); }
#pragma unroll
            for (int j = 0; j < NB; j++) f.ws[0][j] = *(const float*)(sc + 1024 + wave * 256 + (16 * j + r) * 4);
        }
    };
    auto multiply = [&](const Frags& f, float s2) {
        v4f part[NB][MB];
        float xsc[MB], wsc[NB];
        (void)xsc; (void)wsc;
#pragma unroll
        for (int j = 0; j < NB; j++)
#pragma unroll
            for (int b = 0; b < MB; b++) part[j][b] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const int h = s >> 1, d = 2 * (s & 1);
            if constexpr (FORM == FP8X_MX) {
                if (d == 0) {
#pragma unroll
                    for (int b = 0; b < MB; b++) xsc[b] = e8m0_to_f32((f2u(f.xs[0][b]) >> (8 * (q >> 1) + 16 * h)) & 0xffu);
#pragma unroll
                    for (int j = 0; j < NB; j++) wsc[j] = e8m0_to_f32((f2u(f.ws[0][j]) >> (8 * (q >> 1) + 16 * h)) & 0xffu);
                }
            }
            v4i xh[MB];
#pragma unroll
            for (int b = 0; b < MB; b++) xh[b] = widen8<FORM>((uint32_t)f.x[h][b][d], (uint32_t)f.x[h][b][d + 1], xsc[b]);
#pragma unroll
            for (int j = 0; j < NB; j++) {
                const v4i wh = widen8<FORM>((uint32_t)f.w[h][j][d], (uint32_t)f.w[h][j][d + 1], wsc[j]);
#pragma unroll
                for (int b = 0; b < MB; b++) {
                    if constexpr (FORM == FP8X_MX) part[j][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, wh), __builtin_bit_cast(v8bf, xh[b]), part[j][b], 0, 0, 0);
                    else part[j][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, wh), __builtin_bit_cast(v8h, xh[b]), part[j][b], 0, 0, 0);
                }
            }
        }
#pragma unroll
        for (int b = 0; b < MB; b++) {
            const float sc = FORM == FP8X_BLOCK ? f.xs[0][b] * s2 : 1.0f;
#pragma unroll
            for (int j = 0; j < NB; j++)
#pragma unroll
                for (int e = 0; e < 4; e++) acc[j][b][e] = FORM == FP8X_BLOCK ? __builtin_fmaf(part[j][b][e], sc, acc[j][b][e]) : acc[j][b][e] + part[j][b][e];
        }
    };
    if (nt > 0) {
        if constexpr (FORM == FP8X_BLOCK) fetch_scale2(p, t0, nt, nb0, ring + S * TILE + wave * (4 * FS_MOST_BLOCKS));   // (16 NB columns from a multiple of 16 NB on: one scale block)
#pragma unroll
        for (int i = 0; i < S; i++) issue(i, i);
        wait_copies<(S - 1) * CPT>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" : : : "memory");
        Frags f0, f1;
        read(f0, 0);
        int at = 0;
        // tile t + 1 is read while tile t multiplies; tile t + S goes where tile t was, whose fragments every wave holds by then
        auto step = [&](const Frags& now, Frags& then, int t) {
            wait_copies<(S - 2) * CPT>();
            __builtin_amdgcn_s_barrier();
            asm volatile("" : : : "memory");
            issue(t + S, at);
            at = at + 1 < S ? at + 1 : 0;
            read(then, at);
            __builtin_amdgcn_sched_barrier(0);
            float sc = 1.0f;
            if constexpr (FORM == FP8X_BLOCK) sc = *(const float*)(smem + S * TILE + wave * (4 * FS_MOST_BLOCKS) + 4 * t);
            multiply(now, sc);
        };
        for (int t = 0; t < nt; t += 2) {
            step(f0, f1, t);
            if (t + 1 >= nt) break;
            step(f1, f0, t + 1);
        }
        wait_copies<0>();   // (copies past the last tile: none is under way when the workgroup ends)
    }
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
        for (int b = 0; b < MB; b++) fs_store<FORM>(p, m0 + 16 * b + r, n0 + 16 * j + 4 * q, acc[j][b]);
}

// out = epilogue(sum over the K segments, in order, of part[s])
template <int W, int FORM>
__global__ __launch_bounds__(256) void fp8_stream_reduce_kernel(Fp8StreamParams p)
{
    splitk_rows<W>((const float*)p.part, p.splits, (int64_t)p.M * p.N, p.M, p.N, [&](int64_t m, int64_t n0, float (&v)[W]) {
#pragma unroll
        for (int e = 0; e < W; e++) {
            const int64_t n = n0 + e;
            if constexpr (FORM == FP8X_PLAIN) v[e] = (v[e] * p.cs[n * p.cs_stride]) * p.rs[m * p.rs_stride];
            if (p.bias) v[e] = v[e] + p.bias[n];
        }
        store_cols(p.out, p.out_dt, m * p.N + n0, v);
    });
}

template <int FORM>
int launch_reduce(const Fp8StreamParams& p, hipStream_t st)
{
    splitk_launch(p.M, p.N, [&](auto w, dim3 g, dim3 b) { hipLaunchKernelGGL((fp8_stream_reduce_kernel<decltype(w)::value, FORM>), g, b, 0, st, p); });
    return (int)hipGetLastError();
}

template <int MB, int NB, int FORM>
int launch_one(const Fp8StreamParams& p, hipStream_t st)
{
    constexpr int S = fs_stages<MB, NB, FORM>;
    constexpr size_t ring = (size_t)4 * S * fs_tile<MB, NB, FORM> + fs_table<FORM>, sums = (size_t)4 * NB * MB * 1024, lds = ring > sums ? ring : sums;
    static_assert(S >= 2 && lds <= 163840, "the rings of four waves");
    const dim3 grid((unsigned)((p.N + 16 * NB - 1) / (16 * NB)), (unsigned)p.splits, (unsigned)((p.M + 16 * MB - 1) / (16 * MB)));
    auto k = fp8_stream_kernel<MB, NB, FORM, S>;
    static std::atomic<uint64_t> attr_set{0};   // one bit per device: the attribute belongs to the (kernel, device) pair
    if (!device_flag_test(attr_set)) {
        hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return (int)e;
        device_flag_set(attr_set);
    }
    note_route("fp8_stream", p.splits);
    hipLaunchKernelGGL(k, grid, dim3(256), lds, st, p);
    if (hipError_t e = hipGetLastError(); e != hipSuccess || p.splits == 1) return (int)e;
    return launch_reduce<FORM>(p, st);
}
// stages of the wide kernel: two workgroups a CU
template <int MB, int NB, int FORM> constexpr int fw_stages = at_most_8((81920 - fs_table<FORM>) / fw_tile<MB, NB, FORM>);
template <int MB, int NB, int FORM, int KEPT>
int launch_wide_one(const Fp8StreamParams& p, hipStream_t st)
{
    constexpr int S = fw_stages<MB, NB, FORM>;
    constexpr size_t lds = (size_t)S * fw_tile<MB, NB, FORM> + fs_table<FORM>;
    static_assert(S >= 2, "the ring");
    const dim3 grid((unsigned)((p.N + 64 * NB - 1) / (64 * NB)), (unsigned)p.splits, (unsigned)((p.M + 16 * MB - 1) / (16 * MB)));
    auto k = fp8_wide_kernel<MB, NB, FORM, S, KEPT>;
    static std::atomic<uint64_t> attr_set{0};   // one bit per device: the attribute belongs to the (kernel, device) pair
    if (!device_flag_test(attr_set)) {
        hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return (int)e;
        device_flag_set(attr_set);
    }
    note_route("fp8_wide", p.splits);
    hipLaunchKernelGGL(k, grid, dim3(256), lds, st, p);
    if (hipError_t e = hipGetLastError(); e != hipSuccess || p.splits == 1) return (int)e;
    return launch_reduce<FORM>(p, st);
}
template <int FORM>
int launch_form(const Fp8StreamParams& p, const Fp8StreamPlan& pl, hipStream_t st)
{
#define ONE(MB, NB) if (pl.mb == MB && pl.nb == NB) return !pl.wide ? launch_one<MB, NB, FORM>(p, st) : p.kept == 1 ? launch_wide_one<MB, NB, FORM, 1>(p, st) : NB == 1 || p.kept == 2 ? launch_wide_one<MB, NB, FORM, 2>(p, st) : launch_wide_one<MB, NB, FORM, 2 * NB>(p, st);
    ONE(1, 1) ONE(1, 2) ONE(2, 1) ONE(2, 2) ONE(4, 1) ONE(4, 2)
#undef ONE
    if constexpr (FORM != FP8X_BLOCK) {   // (K % 128 == 64 only)
        if (pl.nb == 4) return pl.mb == 1 ? launch_one<1, 4, FORM>(p, st) : pl.mb == 2 ? launch_one<2, 4, FORM>(p, st) : launch_one<4, 4, FORM>(p, st);
    }
    return -1;
}

// Which layout is best: what a launch takes, in us, x2 from memory, fitted to 2700 timed launches of 216 calls (M 4 .. 128, K 1024 .. 16384, N 1024 .. 28000; median error 3 %
// on the wide kernel, 10 % on the other): a start, the K tiles of a workgroup by its row and column blocks -- more than one workgroup a
// CU taking turns --, x2's stream as the other bound, and the second kernel of a K split.
struct StreamCost {
    float start, tile, tile_mn, tile_m, two, reduce, reduce_mb, bw, again;
};
const StreamCost narrow_cost[3] = {   // by Fp8xForm
    {3.5f, 0.116f, 0.039f, 0.108f, 1.88f, 3.2f, 8.0f, 3.5f, 0.0f}, {4.8f, 0.088f, 0.013f, 0.094f, 1.81f, 2.1f, 8.0f, 3.7f, 1.0f}, {3.7f, 0.235f, 0.052f, 0.078f, 1.64f, 3.0f, 8.0f, 3.5f, 0.0f}};
const StreamCost wide_cost[3] = {
    {5.2f, 0.241f, 0.050f, 0.021f, 1.61f, 2.6f, 2.1f, 5.6f, 0.15f}, {5.5f, 0.193f, 0.051f, 0.010f, 1.70f, 1.9f, 2.4f, 5.8f, 0.4f}, {4.7f, 0.296f, 0.055f, 0.025f, 1.73f, 3.0f, 2.1f, 4.3f, 0.33f}};
float turns(int64_t wgs, int per_cu, float two)   // workgroups one after the other, or two at a time
{
    const float w = (float)wgs / 256.0f;
    if (w <= 1.0f) return 1.0f;
    if (per_cu < 2) return (float)((wgs + 255) / 256);
    return w <= 2.0f ? two : two * 0.5f * (0.5f * w + (float)((wgs + 256 * per_cu - 1) / (256 * per_cu)));
}
float stream_us(const StreamCost& c, int mb, int nb, int64_t wgs, int64_t tiles, int64_t slabs, int splits, int per_cu, float x2_mb, float out_m)
{
    const float t = c.tile + c.tile_mn * (float)(mb * nb) + c.tile_m * (float)mb;
    const float cu = (float)tiles * t * turns(wgs, per_cu, c.two), hbm = x2_mb / c.bw * (1.0f + c.again * (float)(slabs - 1));
    const float most = cu > hbm ? cu : hbm, least = cu > hbm ? hbm : cu, q = least / most;
    return c.start + most * (1.0f + 0.19f * q * q * q * q) + (splits > 1 ? c.reduce + c.reduce_mb * (float)splits * out_m : 0.0f);
}
// Whether a call runs here at all: what the chosen layout typically takes, the geometric mean of its time with x2 from memory and with
// x2 in the last-level cache.  Fitted to 12200 launches of 1190 calls in both states (M 1 .. 512, K 1024 .. 18432, N 1024 .. 28672; median error
// 4 %).  `round`: a workgroup's start and end; `few`: x2's rate falls with that power of the share of CUs that have a workgroup.
struct StreamTime {
    float start, tile, tile_mn, tile_m, round, two, bw, again, few, reduce, reduce_mb;
};
const StreamTime narrow_time[3] = {   // by Fp8xForm; its copies and products add up (a workgroup a CU, one ring a wave)
    {1.48f, 0.026f, 0.027f, 0.076f, 2.26f, 1.44f, 9.7f, 0.50f, 0.67f, 0.0f, 0.0f}, {1.44f, 0.010f, 0.027f, 0.051f, 2.2f, 1.33f, 9.4f, 0.61f, 0.58f, 0.0f, 0.0f},
    {1.0f, 0.018f, 0.028f, 0.089f, 2.7f, 1.34f, 6.3f, 0.59f, 0.71f, 0.0f, 0.0f}};
const StreamTime wide_time[3] = {
    {3.26f, 0.204f, 0.063f, 0.004f, 0.87f, 1.6f, 5.9f, 0.67f, 0.0f, 2.3f, 1.44f}, {3.21f, 0.160f, 0.064f, 0.002f, 1.09f, 1.65f, 5.95f, 0.65f, 0.0f, 2.05f, 1.26f},
    {2.84f, 0.221f, 0.075f, 0.017f, 1.16f, 1.61f, 4.9f, 0.37f, 0.48f, 2.7f, 1.43f}};
float stream_typical_us(const StreamTime& c, const Fp8StreamPlan& pl, int64_t wgs, int64_t tiles, int64_t slabs, int per_cu, float x2_mb, float out_m)
{
    const float t = c.tile + c.tile_mn * (float)(pl.mb * pl.nb) + c.tile_m * (float)pl.mb;
    const float cu = turns(wgs, per_cu, c.two) * ((float)tiles * t + c.round);
    const float hbm = x2_mb / c.bw * (1.0f + c.again * (float)(slabs - 1)) * (wgs < 256 ? powf(256.0f / (float)wgs, c.few) : 1.0f);
    const float both = pl.wide ? cbrtf(cu * cu * cu + hbm * hbm * hbm) : cu + hbm;
    return c.start + both + (pl.splits > 1 ? c.reduce + c.reduce_mb * (float)pl.splits * out_m : 0.0f);
}
// The x-in-registers kernel of qmm_fp8_decode.hip on the same terms (900 calls of up to 16 rows, median error 3 %): its workgroups take
// blocks of 16 columns in turns, behind the load of x1 into the waves' registers; idle waves read what others read, which costs no bytes
// from memory.
float decode_typical_us(const QmmDecodePlan& pl, bool mx, int64_t M, int64_t N, float x2_mb, float out_m)
{
    const int64_t cus = 256 / pl.splits, rounds = ((N + 15) / 16 + cus - 1) / cus;
    const float block = mx ? 0.602f : 0.659f, wide = pl.nw == 16 ? (mx ? 2.03f : 1.84f) : 1.0f;
    const float cu = (float)rounds * ((float)pl.nblk * block * wide + (mx ? 0.511f : 0.41f)), hbm = x2_mb / (mx ? 6.43f : 6.85f);
    return (mx ? 2.92f : 2.84f) + (mx ? 4.4e-3f : 2.6e-3f) * (float)(M * pl.nblk * pl.nw) + cbrtf(cu * cu * cu + hbm * hbm * hbm) +
           (pl.splits > 1 ? (mx ? 2.06f : 2.17f) + (mx ? 1.53f : 1.76f) * (float)pl.splits * out_m : 0.0f);
}
// The exact tiles of qmm_fp8_exact.hip on the same terms: their plan's estimate with what it leaves out, and corrected where it is off
// (1066 calls of 65 .. 512 rows, half of them for the fit; median error of the others 2 %; block scales a little high, as the stream kernel's estimate is
// there).  K is cut there from 129 rows, MX from 65.
float tiles_typical_us(int64_t M, int64_t N, int64_t K, Fp8xForm form, bool may_split)
{
    static const struct { float scale, start, out, split; } cost[3] = {   // by Fp8xForm
        {1.05f, 0.2f, 0.21f, 0.7f}, {1.005f, 3.1f, 0.42f, -1.9f}, {1.03f, -2.05f, 0.7f, 1.3f}};
    const auto& c = cost[form];
    const Fp8xPlan pl = fp8x_plan(M, N, K, 1, form, may_split && (M > 128 || form == FP8X_MX));
    const float out_m = (float)M * (float)N * 1e-6f;
    return c.scale * (float)pl.us + c.start + out_m * c.out + (pl.splits > 1 ? c.split : 0.0f);
}
template <int FORM>
constexpr int narrow_per_cu(int mb, int nb)
{
    const int tile = (mb + nb) * 1024 + (FORM == FP8X_BLOCK ? 256 : FORM == FP8X_MX ? 512 : 0);
    const int ring = 4 * at_most_8((163840 - fs_table<FORM>) / 4 / tile) * tile + fs_table<FORM>;
    return 163840 / ring;
}

}  // namespace

// Does a call run here, and how?  (Sizes, types, strides and which operands there are: both phases ask.  x2 K-contiguous, or re-laid
// out so by then.)
//
// Up to 64 rows.  Row / column scales always; block and MX scales with up to 16 rows where the x-in-registers kernel of qmm_fp8_decode.hip
// is not ahead by the estimates above (x2 from memory, there and here: 16 x 7168 x 18432 37 and 35 us, MX 3 x 6272 x 19456 33 and 41,
// 1 x 1792 x 8192 7.8 and 9.2, but 8 x 3200 x 1920 9.0 and 7.9; 8 x 9856 x 23040, which it cuts, 61 and 44).
//
// From 65 to 512 rows, in slabs of 64: products that leave most of the exact tiles without a CU's worth of work, by the estimates
// (typical times there and here, MX 65 x 2048 x 2304 13.4 and 10.1 us, 128 x 1664 x 1472 15.2 and 8.9, 128 x 13568 x 8960 52 and 67,
// 96 x 7424 x 18816 55 and 77; row / column scales 181 x 2560 x 2368 16.4 and 11.1, 114 x 11520 x 22208 89 and 108; block scales
// 405 x 1664 x 3848 24.2 and 18.9; of 1066 calls 6 run 5 % longer than on the other side, the worst 1.13 times.  With the corrections of the tiles'
// former plan 31 did, the worst 1.29 times: row / column scales 109 x 16640 x 15253 91 here and 106 there, MX 114 x 2944 x 4757 18.2 and
// 19.5, block scales 194 x 6144 x 1472 16.9 and 18.8).  A last half K tile runs on padded copies there: here up to so many multiplications above 128 rows (row /
// column scales 246 x 12224 x 2560 76 and 49).
constexpr int64_t FS_MANY_ROWS_TAIL = 3200000000, FS_MANY_ROWS_TAIL_PLAIN = 12000000000;
bool fp8_stream_plan(const OpsnnQmmArgs& a, Fp8xForm form, bool may_split, Fp8StreamPlan& pl)
{
    if (a.x1_dtype != DT_E4M3 || a.x2_dtype != DT_E4M3 || a.batch != 1 || a.force_variant != 0) return false;
    if (a.out_dtype != DT_BF16 && a.out_dtype != DT_F16 && a.out_dtype != DT_F32) return false;
    if (a.M > 512 || a.N < 256 || a.K < 128 || a.K % 64 != 0 || a.K >= (1ll << 30) || a.N >= (1ll << 30)) return false;
    if (a.M > 128 && (a.K < 1024 || (a.K % 128 && a.M * a.N * a.K > (form == FP8X_PLAIN ? FS_MANY_ROWS_TAIL_PLAIN : FS_MANY_ROWS_TAIL)))) return false;
    const int64_t ldb = a.x2.row_stride == 1 ? a.x2.col_stride : a.K;
    // (32-bit lane offsets: from the first row of x1 and of its scales, from the workgroup's first column of x2)
    auto offsets_ok = [](int64_t rows, int64_t bytes) { return bytes >= 0 && bytes < (1ll << 31) / rows; };
    if (!offsets_ok(a.M, a.x1.row_stride) || ldb < 0 || ldb >= (1ll << 24)) return false;
    if (form == FP8X_BLOCK) {
        if (a.K % 128 != 0 || a.bias || a.gsK != 128 || a.gsN != 128 || (a.gsM != 1 && a.gsM != 128)) return false;
        if (!offsets_ok(a.M, 4 * a.x1_scale_mat.row_stride) || a.x2_scale_mat.row_stride < 0 || a.x2_scale_mat.row_stride >= (1ll << 20)) return false;
    } else if (form == FP8X_PLAIN) {
        if (!a.x1_scale || !a.x2_scale || a.x2_scale_dtype != DT_F32 || (a.bias && a.bias_dtype != DT_F32)) return false;
        if (a.x1_scale_len == 1 && a.x2_scale_len == 1 && !a.bias) return false;   // (that case merges and truncates the scales)
    } else {
        if ((a.bias && a.bias_dtype != DT_F32) || !offsets_ok(a.M, a.x1_scale_mat.row_stride) || a.x2_scale_mat.row_stride < 0) return false;
        if (a.x2_scale_mat.row_stride >= (1ll << 24)) return false;
    }
    const int mb = a.M <= 16 ? 1 : a.M <= 32 ? 2 : 4;
    const int64_t slabs = (a.M + 16 * mb - 1) / (16 * mb), units = (a.K + 127) / 128;
    const bool whole = a.K % 128 == 0;
    const float x2_mb = (float)a.N * (float)a.K * 1e-6f, out_m = (float)a.M * (float)a.N * 1e-6f;
    pl.mb = mb;
    float best = 1e30f;
    int64_t wgs = 0, k_tiles = 0;   // of the best so far
    int cu_wgs = 1;
    auto consider = [&](bool wide, int nb, int splits, int per_cu) {
        const int64_t strips = (a.N + (wide ? 64 : 16) * nb - 1) / ((wide ? 64 : 16) * nb), seg = (units + splits - 1) / splits;
        const int64_t per_wave = wide ? seg : (seg + 3) / 4;
        if (splits > 1 && (!may_split || units < 4 * splits)) return;
        if (form == FP8X_BLOCK && per_wave > FS_MOST_BLOCKS) return;
        // (partial sums of a row that is no whole number of quads count twice: their stores straddle lines, and where they did not count so,
        // 19 of 200 such calls of up to 64 rows were cut otherwise and took 1.026 times as long, fp8 and weight-only together)
        const float us = stream_us(wide ? wide_cost[form] : narrow_cost[form], mb, nb, strips * splits * slabs, wide ? seg : 2 * per_wave, slabs, splits, per_cu, x2_mb, a.N % 4 ? 2.0f * out_m : out_m);
        if (us < best) { best = us; pl.wide = wide; pl.nb = nb; pl.splits = splits; wgs = strips * splits * slabs; k_tiles = wide ? seg : 2 * per_wave; cu_wgs = per_cu; }
    };
    // the narrow kernel where one round of workgroups is enough, the wide one for the rest; a last half K tile is the narrow one's
    static const int steps[8] = {1, 2, 3, 4, 6, 8, 12, 16};
    for (int nb = 1; nb <= 2; nb++) {
        const int per_cu = form == FP8X_BLOCK ? narrow_per_cu<FP8X_BLOCK>(mb, nb) : form == FP8X_PLAIN ? narrow_per_cu<FP8X_PLAIN>(mb, nb) : narrow_per_cu<FP8X_MX>(mb, nb);
        if (!whole || (a.N + 16 * nb - 1) / (16 * nb) * slabs <= 256 * per_cu) consider(false, nb, 1, per_cu);
        for (int i = 0; whole && i < 8; i++) consider(true, nb, steps[i], 2);
    }
    for (int i = 0; !whole && i < 6; i++) consider(false, 4, steps[i], 1);
    if (best >= 1e30f) return false;
    if (whole && (a.M > 64 || (a.M <= 16 && form != FP8X_PLAIN))) {
        const float out = a.N % 4 && a.M <= 64 ? 2.0f * out_m : out_m, here = stream_typical_us((pl.wide ? wide_time : narrow_time)[form], pl, wgs, k_tiles, slabs, cu_wgs, x2_mb, out);
        if (a.M > 64) return here <= tiles_typical_us(a.M, a.N, a.K, form, may_split);
        // (1.04: this kernel's estimate is 2 to 10 % high up to 16 rows.  Of 700 calls drawn after the fit 33 are 5 % slower or more than on the other
        // kernel, of 900 without x1's load and this factor 78.)
        if (QmmDecodePlan dp; qmm_decode_plan(a.K, may_split, dp) && 1.04f * decode_typical_us(dp, form == FP8X_MX, a.M, a.N, x2_mb, out) < here) return false;
    }
    return true;
}

int launch_fp8_stream(const OpsnnQmmArgs& a, Fp8xForm form, SplitK sk, hipStream_t st)
{
    Fp8StreamPlan pl;
    // (the caller asked for the 8-bit instruction, which has no fp32 outputs but for MX)
    if (a.M > 128 && a.K % 128 == 0 && (a.out_dtype != DT_F32 || form == FP8X_MX) && opsnnGetFp8Fast()) return OPSNN_NOT_TAKEN;
    if (!fp8_stream_plan(a, form, true, pl)) return OPSNN_NOT_TAKEN;
    // (no partial sums, or laid out for other segments: a call that another layout of its operands has changed on the way)
    if (pl.splits > 1 && (!sk.part || sk.splits < pl.splits) && !fp8_stream_plan(a, form, false, pl)) return OPSNN_NOT_TAKEN;
    const int splits = pl.splits;
    if (a.x1.col_stride != 1 || a.x2.row_stride != 1) return OPSNN_NOT_TAKEN;
    Fp8StreamParams p{};
    p.a = (const uint8_t*)a.x1.ptr; p.b = (const uint8_t*)a.x2.ptr; p.lda = a.x1.row_stride; p.ldb = a.x2.col_stride;
    if (((uintptr_t)p.a | (uintptr_t)p.b | (uint64_t)p.lda | (uint64_t)p.ldb) % 16) return OPSNN_NOT_TAKEN;
    p.out = a.out; p.out_dt = a.out_dtype; p.M = (int)a.M; p.N = (int)a.N; p.tiles = (int)(a.K / 64); p.splits = splits;
    p.part = sk.part; p.bias = (const float*)a.bias;
    p.kept = a.M <= 64 ? weight_kept_share(a.N * a.K) : 1;
    if (form == FP8X_BLOCK) {
        p.s1 = (const float*)a.x1_scale_mat.ptr; p.s1_rs = a.x1_scale_mat.row_stride; p.s1_cs = a.x1_scale_mat.col_stride;
        p.s2 = (const float*)a.x2_scale_mat.ptr; p.s2_rs = a.x2_scale_mat.row_stride; p.s2_cs = a.x2_scale_mat.col_stride;
        p.gsM = (int)a.gsM;
        if (((uintptr_t)p.s1 | (uintptr_t)p.s2) % 4) return OPSNN_NOT_TAKEN;
        return launch_form<FP8X_BLOCK>(p, pl, st);
    }
    if (form == FP8X_PLAIN) {
        p.rs = (const float*)a.x1_scale; p.cs = (const float*)a.x2_scale; p.rs_stride = a.x1_scale_len == 1 ? 0 : 1; p.cs_stride = a.x2_scale_len == 1 ? 0 : 1;
        return launch_form<FP8X_PLAIN>(p, pl, st);
    }
    p.sa = (const uint8_t*)a.x1_scale_mat.ptr; p.sa_rs = a.x1_scale_mat.row_stride;
    p.sb = (const uint8_t*)a.x2_scale_mat.ptr; p.sb_rs = a.x2_scale_mat.row_stride;
    if (a.x1_scale_mat.col_stride != 2 || a.x2_scale_mat.col_stride != 2) return OPSNN_NOT_TAKEN;   // [rows, K / 64, 2]: a row's bytes contiguous
    if (((uintptr_t)p.sa | (uintptr_t)p.sb | (uint64_t)p.sa_rs | (uint64_t)p.sb_rs) % (pl.wide ? 4 : 2)) return OPSNN_NOT_TAKEN;
    return launch_form<FP8X_MX>(p, pl, st);
}

}  // namespace opsnn
