// Weight-only matmul, up to 1024 rows of x, either storage of the weight ([N, K] and [K, N]), any group that is a power of two from 32.
//
// What bounded these calls (17 .. 64 rows on the kernels of wq_nk.hip, wq_kn.hip and wqmm_stream.hip.h, more rows on the dequantising
// pass of wq_dense.hip): operands loaded straight into the layout of the matrix instructions, 16 rows per 16 lanes, take 66 clocks a KB
// in the memory pipeline of a CU, twice what the same bytes take with neighbouring lanes side by side; and a dequantised copy of the
// weight is four times its bytes, written and read.  So weight and x travel global -> LDS as they lie, 16 bytes a lane, asynchronously,
// in K tiles of 128 for 128 columns and 16 MB rows, through a ring of as many stages as the LDS holds, one barrier a tile, and every
// weight is dequantised once per 16 MB rows, in registers.
//
// Eight waves: two halves of the columns times four steps of 32 k.  A wave multiplies 64 columns by all rows with 32 x 32 x 16 products,
// each fragment of x for both column blocks; the sums over k meet in LDS at the end, in order.  (One row block: four quarters of the
// columns times two steps of 64 k, 16 x 16 x 32 products.)  blockIdx.y cuts K further (fp32 partial sums, added in order by
// wq_splitk_reduce_kernel), blockIdx.z takes further slabs of 16 MB rows.  The scales of the workgroup's columns lie in LDS as a table,
// laid down once: a compiler's load in the loop would be waited for with every copy under way.
//
// What bounds it is the issue of vector instructions, from 33 rows against a wide N also the power: 64 x 8192 x 28672 fp16 runs at 1.96 GHz
// (2.38 with x zero).  Two waves a SIMD issue a packed fp16 operation, permute, shift or conversion in 2.15 ns and an fp32 or bit operation
// in 1.75; a 16 x 16 x 32 product stands in their way for 4 ns, a 32 x 32 x 16 one, twice the work, for as long.  So: the large products;
// operands in k order, so that x needs no permutation (three operations more for eight codes of fp16 x int4, four fewer for a fragment of
// x); [K, N] storage through the LDS reads that transpose, which deliver what the [N, K] form reads, where pairs of rows were
// spliced before; bf16 x int4 without offsets through a conversion that takes two codes at a time.  Sixteen waves a workgroup, copies from
// waves of their own, and reads and copies spread between the products changed nothing (57.6, 57.5, 58.6 us for 57.8, 64 x 8192 x 28672).
//
// LDS rows, conflict-free for the reads below: x 256 bytes, 16-byte chunk c of row r at c ^ (r % 16); [N, K] weights 64 bytes (4 bits),
// c ^ (r / 4 % 4), or 128, c ^ (r / 2 % 8); [K, N] weights, a row of k each, 64 bytes, c ^ (k / 4 % 4), or 128, c ^ 2 (k / 2 % 4).
// A [K, N] weight whose rows are whole dwords but not 16-byte pieces (N a multiple of 8 with 4 bits, of 4 with 8) is copied a dword a lane, four
// copies for one (4 bits) and eight for two (8 bits) a wave and tile.  0.05 us a tile (4 bits) and 0.1 (8).
//
// Measured, before these products and reads and with them, the weight in turn from three buffers: 121 drawn calls of 1 .. 512 rows 1.058 times as
// fast, none slower by more than 2 %; bf16 x int4 499 x 13632 x 3052 77 -> 64 us, 129 x 14912 x 3328 41 -> 35; fp16 64 x 16384 x 5120 91 -> 81
// (the kernel alone), [K, N] bf16 4 x 2240 x 4224 10.4 -> 8.9.  Against the kernels before this one: [K, N] int4, 110 x 11008 x 24768 fp16 346 ->
// 126 us, 73 x 6656 x 2752 34.9 -> 19.0, int8 67 x 3840 x 12864 65 -> 30; [N, K] int4 57 x 9856 x 24349 98 -> 63, int8 118 x 14336 x 8512 bf16 135 -> 58.
#include "launch.h"
#include "wq_cost.h"
#include "wqmm_stream.hip.h"

extern "C" int opsnn_wq_tile_min();   // dispatch.hip
extern "C" int opsnn_wq_narrow_slabs();
namespace opsnn {
bool wq_nk_wanted(const OpsnnWqmmArgs& a, uint64_t* workspace);   // wq_nk.hip
double wq_nk_typical_us(const OpsnnWqmmArgs& a);
bool wq_kn_wanted(const OpsnnWqmmArgs& a);   // wq_kn.hip
double wq_kn_typical_us(const OpsnnWqmmArgs& a);
double wq_many_rows_typical_us(const OpsnnWqmmArgs& a);   // wq_dense.hip
bool weight_cache_on();                                 // weight_cache.hip
const void* weight_cache_get(const void* src, int64_t K, int64_t N, int bits, int64_t nb, hipStream_t st);
namespace {

constexpr int WW_COLS = 128, WW_KT = 128;   // columns of a workgroup, k of a tile

// 8 codes of consecutive k (4 bits: one dword, 8 bits: two) -> an operand of the matrix instructions, in k order.  The arithmetic and its
// two roundings are those of dequant8 in wqmm_stream.hip.h.
struct WwConst {
    uint32_t mask, flip;   // fp16, 4 bits: the low nibble of the low half, the high one of the high half; their sign bits under the exponent of 1024.0
    h2 unit, base;
};
__device__ __forceinline__ WwConst ww_const()
{
    WwConst c = {0x00f0000fu, 0x64806408u, {(_Float16)1.0f, (_Float16)0.0625f}, {(_Float16)-1032.0f, (_Float16)-72.0f}};
    asm volatile("" : "+v"(c.mask), "+v"(c.flip), "+v"(c.unit), "+v"(c.base));   // (registers: the three-operand forms take no literals)
    return c;
}
// E4M3 (bf16, 4 bits, no offset): by way of e4m3 codes, for scales below 2^125
template <int XDT, int WBITS, bool HAS_OFF, bool E4M3>
__device__ __forceinline__ v4i ww_dequant(const uint32_t* w, uint32_t so, const WwConst& dc)
{
    v4i r;
    if constexpr (XDT == DT_F16) {
        const _Float16 sh = __builtin_bit_cast(_Float16, (uint16_t)so), oh = __builtin_bit_cast(_Float16, (uint16_t)(so >> 16));
#pragma unroll
        for (int i = 0; i < 4; i++) {
            h2 t;
            if constexpr (WBITS == 4) {   // byte i in both halves: 1024 + (w + 8) of its low nibble, 1024 + 16 (w + 8) of its high one
                const uint32_t b = __builtin_amdgcn_perm(w[0], w[0], 0x0c000c00u | (uint32_t)i | (uint32_t)i << 16);
                t = __builtin_elementwise_fma(__builtin_bit_cast(h2, (b & dc.mask) ^ dc.flip), dc.unit, dc.base);   // exact
            } else {
                const h2 c1152 = {(_Float16)-1152.0f, (_Float16)-1152.0f};
                t = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, w[i >> 1] ^ 0x80808080u, i & 1 ? 0x04030402u : 0x04010400u)) + c1152;
            }
            if constexpr (HAS_OFF) t = t + (h2){oh, oh};
            r[i] = (int)u32(t * (h2){sh, sh});
        }
    } else {
        const float sc = bf16_to_f32((uint16_t)so), off = bf16_to_f32((uint16_t)(so >> 16));
        float v[8];
        if constexpr (E4M3) {
            // w + 8 in a byte reads as the e4m3 value 2^-9 (w + 8): two conversions at a time, and the fma's (w + 8) s - 8 s is w s
            const uint32_t lo = (w[0] & 0x0f0f0f0fu) ^ 0x08080808u, hi = ((w[0] >> 4) & 0x0f0f0f0fu) ^ 0x08080808u;
            const v2f l0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(lo, 512.0f, false), l1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(lo, 512.0f, true);
            const v2f h0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(hi, 512.0f, false), h1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(hi, 512.0f, true);
            const float s8 = -8.0f * sc;
            v[0] = __builtin_fmaf(l0[0], sc, s8); v[1] = __builtin_fmaf(h0[0], sc, s8); v[2] = __builtin_fmaf(l0[1], sc, s8); v[3] = __builtin_fmaf(h0[1], sc, s8);
            v[4] = __builtin_fmaf(l1[0], sc, s8); v[5] = __builtin_fmaf(h1[0], sc, s8); v[6] = __builtin_fmaf(l1[1], sc, s8); v[7] = __builtin_fmaf(h1[1], sc, s8);
        } else {
            // (4 bits: a nibble at the top of its byte, 16 times the weight, converts as it lies)
            const uint32_t odd = w[0] & 0xf0f0f0f0u, even = (w[0] << 4) & 0xf0f0f0f0u;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float c = WBITS == 4 ? (float)((int)((i & 1 ? odd : even) << (24 - 8 * (i >> 1))) >> 24) : (float)((int)(w[i >> 2] << (24 - 8 * (i & 3))) >> 24);
                v[i] = HAS_OFF ? __builtin_fmaf(c, WBITS == 4 ? 0.0625f : 1.0f, off) : c;
            }
            if constexpr (HAS_OFF) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const uint32_t pk = pack2_bf16((v2f){v[2 * i], v[2 * i + 1]});
                    v[2 * i] = u2f(pk << 16);
                    v[2 * i + 1] = u2f(pk & 0xffff0000u);
                }
            }
            const float unit = WBITS == 4 && !HAS_OFF ? 0.0625f * sc : sc;
#pragma unroll
            for (int i = 0; i < 8; i++) v[i] = v[i] * unit;
        }
#pragma unroll
        for (int i = 0; i < 4; i++) r[i] = (int)pack2_bf16((v2f){v[2 * i], v[2 * i + 1]});
    }
    return r;
}

// Reads that transpose (lane layouts checked on the chip): of sixteen lanes, each at 8 bytes, lane l gets nibble l of all sixteen; or, in
// pairs at 16 bytes of a row, byte l of the eight rows.
typedef __attribute__((address_space(3))) v2i LdsV2i;
__device__ __forceinline__ v2i lds_read_tr4(const char* at) { return __builtin_amdgcn_ds_read_tr4_b64_v2i32((LdsV2i*)at); }
__device__ __forceinline__ v2i lds_read_tr8(const char* at) { return __builtin_amdgcn_ds_read_tr8_b64_v2i32((LdsV2i*)at); }

// bytes of a tile, stages of the ring, bytes of the ring (at least what the sums need at the end), groups that the table has room for
constexpr int ww_tile(int wbits, int mb) { return mb * 4096 + WW_COLS * WW_KT * wbits / 8; }
constexpr int ww_stages(int wbits, int mb)
{
    return wbits == 4 ? (mb <= 2 ? 6 : mb <= 4 ? 4 : 3) : (mb <= 4 ? 4 : 3);
}
constexpr int ww_ring(int wbits, int mb) { const int a = ww_tile(wbits, mb) * ww_stages(wbits, mb); return a > 65536 ? a : 65536; }
constexpr int ww_groups(int wbits, int mb) { return (163840 - ww_ring(wbits, mb)) / (WW_COLS * 4); }

// [N, K] storage; [K, N] storage with rows of whole 16-byte pieces; of whole dwords
enum WwStorage { WW_NK, WW_KN, WW_KN4 };

template <int XDT, int WBITS, int MB, bool HAS_OFF, int STORAGE>
__global__ __launch_bounds__(512, 1) void wq_wide_kernel(WqParams p, int tiles, int splits, int gmax)
{
    constexpr bool BIG = MB >= 2;                                            // 32 x 32 x 16, or 16 x 16 x 32
    constexpr int LC = BIG ? 32 : 16, RB = BIG ? MB / 2 : MB, CB = 2;         // columns and rows of a block, row and column blocks of a wave
    constexpr int WN = WW_COLS / (CB * LC), KW = 8 / WN, KS = WW_KT / KW;    // waves across columns and k, k of a wave's step
    constexpr int E4 = BIG ? 4 : 1;                                          // quads of a block's sums that a lane has
    constexpr int TILE = ww_tile(WBITS, MB), S = ww_stages(WBITS, MB);
    constexpr bool KN = STORAGE != WW_NK;
    constexpr int WP = STORAGE == WW_KN4 ? 4 : 16;                                       // bytes of a lane's copy of the weight
    constexpr int XC = MB > 2 ? MB / 2 : 1, WC = WBITS / 4 * (16 / WP), CPT = XC + WC;   // copies per wave and tile
    constexpr int WROW = WW_KT * WBITS / 8;                                  // bytes of a weight row in a tile
    typedef std::conditional_t<BIG, v16f, v4f> Acc;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave % WN, kw = wave / WN;
    const int c = lane % LC, qh = lane / LC;
    const int Ni = (int)p.N, Ki = (int)p.K, Mi = (int)p.M;
    const int n0 = (int)blockIdx.x * WW_COLS, m0 = (int)blockIdx.z * (16 * MB);
    const int t0 = (int)((int64_t)blockIdx.y * tiles / splits), nt = (int)((int64_t)(blockIdx.y + 1) * tiles / splits) - t0;
    const int gshift = p.group_shift;
    auto group_at = [&](int k) { return k >> gshift; };
    auto base_of = [&](int t) { const int k = (t0 + t) * WW_KT; return k + WW_KT <= Ki ? k : Ki - WW_KT; };   // (a last, partial tile starts early)
    const int g_lo = group_at(base_of(0)), g_all = group_at(Ki - 1);

    // copies: x rows of 256 bytes, four per copy; weight rows of 64 (4 bits) or 128 bytes, sixteen or eight per copy
    uint32_t xo[XC], wo[WC];
#pragma unroll
    for (int i = 0; i < XC; i++) {
        const int row = ((wave * XC + i) * 4 + (lane >> 4)) % (16 * MB), m = m0 + row < Mi ? m0 + row : Mi - 1;
        xo[i] = (uint32_t)(m - m0) * (uint32_t)(2 * Ki) + 16 * ((lane & 15) ^ (row & 15));
    }
#pragma unroll
    for (int i = 0; i < WC; i++) {
        const int piece = (wave * WC + i) * 64 + lane, row = piece / (WROW / WP), b = piece % (WROW / WP) * WP;   // a column, or a row of k; byte of the LDS row
        if constexpr (KN) {
            const int at = (b ^ 16 * (WBITS == 4 ? (row >> 2) & 3 : 2 * ((row >> 1) & 3))), last = (Ni - n0) * WBITS / 8 - WP;
            wo[i] = (uint32_t)row * (uint32_t)p.ldw + (at < last ? at : last);
        } else {
            const int n = n0 + row < Ni ? row : Ni - 1 - n0;
            wo[i] = (uint32_t)n * (uint32_t)p.ldw + (b ^ 16 * (WBITS == 4 ? (row >> 2) & 3 : (row >> 1) & 7));
        }
    }
    const char* const xbase = (const char*)(p.x + (int64_t)m0 * Ki);
    const char* const wbase = (const char*)(KN ? p.w + (int64_t)n0 * WBITS / 8 : p.w + (int64_t)n0 * p.ldw);
    const uint32_t ring = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)smem;
    // (bases only grow, so that the last one bounds them all: past the end it is fetched and read again)
    const int k_last = __builtin_amdgcn_readfirstlane(base_of(nt - 1));
    int k_issue = __builtin_amdgcn_readfirstlane(t0 * WW_KT), k_read = k_issue;
    auto issue = [&](int stage) {
        const int64_t k = k_issue < k_last ? k_issue : k_last;
        k_issue += WW_KT;
        const uint32_t at = __builtin_amdgcn_readfirstlane(ring + stage * TILE);
#pragma unroll
        for (int i = 0; i < WC; i++) {
            if constexpr (WP == 16) copy16_sbase(wbase + (KN ? k * p.ldw : k * WBITS / 8), wo[i], at + MB * 4096 + (wave * WC + i) * 1024);
            else copy4_sbase(wbase + k * p.ldw, wo[i], at + MB * 4096 + (wave * WC + i) * 256);
        }
#pragma unroll
        for (int i = 0; i < XC; i++) copy16_sbase(xbase + k * 2, xo[i], at + ((wave * XC + i) * 1024) % (MB * 4096));
    };

    Acc acc[CB][RB] = {};
    constexpr bool PERMUTE = !BIG && XDT == DT_F16 && WBITS == 4;   // one row block: four permutes for a fragment of x cost less than three more for each of its two operands
    constexpr bool MAY_E4M3 = XDT == DT_BF16 && WBITS == 4 && !HAS_OFF;
    const WwConst dqc = ww_const();
    const DqConst dqp = make_dq_const();
    uint32_t* const tab = (uint32_t*)(smem + ww_ring(WBITS, MB));
    // A lane multiplies k = KS kw + 16 qh .. + 15 of its columns and rows, eight at a time.
    struct Frags {
        v4i x[RB][2];
        uint32_t w[CB][WBITS / 2];
        uint32_t so[CB];
    };
    const int ck = (KS * kw + 16 * qh) / 8;   // in pieces of 8 k
    auto read = [&](Frags& f, int stage) {
        const int k = k_read < k_last ? k_read : k_last;
        k_read += WW_KT;
        const char* const at = smem + stage * TILE;
        const char* const wat = at + MB * 4096;
#pragma unroll
        for (int b = 0; b < RB; b++)
#pragma unroll
            for (int i = 0; i < 2; i++) f.x[b][i] = *(const v4i*)(at + (LC * b + c) * 256 + 16 * ((ck + i) ^ (c & 15)));
#pragma unroll
        for (int j = 0; j < CB; j++) {
            const int col = (wn * CB + j) * LC + c;
            if constexpr (!KN && WBITS == 4) __builtin_memcpy(f.w[j], __builtin_assume_aligned(wat + col * WROW + 16 * ((ck >> 2) ^ ((col >> 2) & 3)) + 4 * (ck & 2), 8), 8);
            else if constexpr (!KN) __builtin_memcpy(f.w[j], __builtin_assume_aligned(wat + col * WROW + 16 * ((ck >> 1) ^ ((col >> 1) & 7)), 16), 16);
            else {
                // the transposing reads: sixteen lanes point at 16 k x 16 columns of 4 bits (8 k of 8 bits), and each gets a column's codes
                const int n = (wn * CB + j) * LC + (BIG ? lane & 16 : 0);
                if constexpr (WBITS == 4) {
                    const int row = 8 * ck + (lane & 15);
                    const v2i v = lds_read_tr4(wat + row * 64 + 16 * ((n >> 5) ^ ((row >> 2) & 3)) + ((n >> 1) & 8));
                    f.w[j][0] = (uint32_t)v[0]; f.w[j][1] = (uint32_t)v[1];
                } else {
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        const int row = 8 * (ck + i) + ((lane & 15) >> 1);
                        const v2i v = lds_read_tr8(wat + row * 128 + 16 * ((n >> 4) ^ (2 * ((row >> 1) & 3))) + 8 * (lane & 1));
                        f.w[j][2 * i] = (uint32_t)v[0]; f.w[j][2 * i + 1] = (uint32_t)v[1];
                    }
                }
            }
            f.so[j] = tab[(group_at(k + 8 * ck) - g_lo) * WW_COLS + col];
        }
    };
    auto multiply = [&](const Frags& f, auto e4m3, bool part, bool counts) {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            v4i xf[RB];
#pragma unroll
            for (int b = 0; b < RB; b++) {
                xf[b] = f.x[b][i];
                if constexpr (PERMUTE) {   // halves [0..7] -> [0,4,1,5,2,6,3,7]
                    const uint32_t a0 = (uint32_t)xf[b][0], a1 = (uint32_t)xf[b][1], a2 = (uint32_t)xf[b][2], a3 = (uint32_t)xf[b][3];
                    xf[b] = (v4i){(int)__builtin_amdgcn_perm(a2, a0, 0x05040100u), (int)__builtin_amdgcn_perm(a2, a0, 0x07060302u),
                                  (int)__builtin_amdgcn_perm(a3, a1, 0x05040100u), (int)__builtin_amdgcn_perm(a3, a1, 0x07060302u)};
                }
            }
#pragma unroll
            for (int j = 0; j < CB; j++) {
                v4i a;
                if constexpr (PERMUTE) a = dequant8<XDT, WBITS, HAS_OFF>((v4i){(int)f.w[j][i], 0, 0, 0}, 0, (uint16_t)f.so[j], (uint16_t)(f.so[j] >> 16), dqp);
                else a = ww_dequant<XDT, WBITS, HAS_OFF, decltype(e4m3)::value>(f.w[j] + i * (WBITS / 4), f.so[j], dqc);
                if (part) a = counts ? a : (v4i){0, 0, 0, 0};
#pragma unroll
                for (int b = 0; b < RB; b++) {
                    const v4i x = part && !counts ? (v4i){0, 0, 0, 0} : xf[b];
                    if constexpr (BIG && XDT == DT_F16) acc[j][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, x), acc[j][b], 0, 0, 0);
                    else if constexpr (BIG) acc[j][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, x), acc[j][b], 0, 0, 0);
                    else if constexpr (XDT == DT_F16) acc[j][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, x), acc[j][b], 0, 0, 0);
                    else acc[j][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, x), acc[j][b], 0, 0, 0);
                }
            }
        }
    };
    // Scale table: word (group - g_lo, column) = scale | offset << 16.  Eight at a time where they lie so -- along the groups of a column
    // (by_group) or along the columns --, fetched in front of the first copies and put down behind them.
    const bool by_group = p.s_rs == 1;
    const bool wide = (by_group ? p.s_cs : p.s_rs) % 8 == 0 && (by_group || p.s_cs == 1) && ((uintptr_t)p.scale | (uintptr_t)(HAS_OFF ? p.offset : nullptr)) % 16 == 0;
    const int t_col = by_group ? tid >> 2 : 8 * (tid & 15), t_g = by_group ? (g_lo & ~7) + 8 * (tid & 3) : g_lo + (tid >> 4);
    struct Eight { uint16_t s[8], o[8]; };
    auto load8 = [&](Eight& v, int i) {
        const int g = t_g + 32 * i, n = n0 + t_col;
        const bool all = by_group ? g + 7 <= g_all && n < Ni : g <= g_all && n + 7 < Ni;
        if (wide && all) {
            const int64_t at = (int64_t)g * p.s_rs + (int64_t)n * p.s_cs;
            *(v4i*)v.s = *(const v4i*)(p.scale + at);
            if constexpr (HAS_OFF) *(v4i*)v.o = *(const v4i*)(p.offset + at);
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int ge = g + (by_group ? e : 0), ne = n + (by_group ? 0 : e);
                const int64_t at = (int64_t)(ge < g_all ? ge : g_all) * p.s_rs + (int64_t)(ne < Ni ? ne : Ni - 1) * p.s_cs;
                v.s[e] = p.scale[at];
                if constexpr (HAS_OFF) v.o[e] = p.offset[at];
            }
        }
    };
    // Without offsets the upper halves of the table's words are free.  Those of the first eight hold a flag of each wave: the table can be as large as
    // the LDS has room for (212 x 10112 x 12096 in groups of 128 fills it; with the flags behind it K had to be cut in four: bf16 in [K, N] storage 97.8 us so, 102.5 cut).
    typedef uint16_t __attribute__((may_alias)) Half;
    Half* const halves = (Half*)tab;
    bool large = false;   // a scale from 2^125 on, an infinity or NaN
    auto store8 = [&](const Eight& v, int i) {
        const int g = t_g + 32 * i - g_lo;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            if constexpr (MAY_E4M3) large = large || (v.s[e] & 0x7f80) >= 0x7e00;
            const int ge = g + (by_group ? e : 0), ne = t_col + (by_group ? 0 : e);
            if (ge < 0 || ge >= gmax) continue;
            if constexpr (MAY_E4M3) halves[2 * (ge * WW_COLS + ne)] = v.s[e];
            else tab[ge * WW_COLS + ne] = HAS_OFF ? v.s[e] | (uint32_t)v.o[e] << 16 : v.s[e];
        }
    };
    {
        Eight v0, v1;
        for (int i = 2; 32 * i < gmax + 7; i++) { load8(v0, i); store8(v0, i); }
        load8(v0, 0);
        if (32 < gmax + 7) load8(v1, 1);
        wait_copies<0>();   // (these loads, for the compiler)
#pragma unroll
        for (int i = 0; i < S; i++) issue(i);
        store8(v0, 0);
        if (32 < gmax + 7) store8(v1, 1);
    }
    if constexpr (MAY_E4M3) {
        const uint64_t any = __ballot(large);
        if (lane == 0) halves[2 * wave + 1] = any != 0;
    }
    wait_copies<(S - 1) * CPT>();
    __syncthreads();
    // (a last, partial tile: what lies in front of it was counted with the one before)
    const bool part = (t0 + nt) * WW_KT > Ki, counts = base_of(nt - 1) + 8 * ck >= (t0 + nt - 1) * WW_KT;
    auto walk = [&](auto e4m3) {
        if constexpr (MB <= 4) {
            Frags f0, f1;
            read(f0, 0);
            int t = 0, at = 0;
            // tile t + 1 is read while tile t multiplies; tile t + S goes where tile t was, whose fragments every wave holds by then
            auto step = [&](const Frags& now, Frags& then) {
                wait_copies<(S - 2) * CPT>();
                __builtin_amdgcn_s_barrier();
                asm volatile("" : : : "memory");
                issue(at);
                at = at + 1 < S ? at + 1 : 0;
                read(then, at);
                __builtin_amdgcn_sched_barrier(0);
                multiply(now, e4m3, false, true);
            };
            for (; t + 2 < nt; t += 2) {
                step(f0, f1);
                step(f1, f0);
            }
            if (t + 1 < nt) {
                step(f0, f1);
                multiply(f1, e4m3, part, counts);
            } else multiply(f0, e4m3, part, counts);
        } else {   // (no registers for a second set of fragments: tile t + S - 1 goes where tile t - 1 was)
            Frags f;
            int at = 0, free = S - 1;
            for (int t = 0; t < nt; t++) {
                wait_copies<(S - 2) * CPT>();
                __builtin_amdgcn_s_barrier();
                asm volatile("" : : : "memory");
                if (t > 0) issue(free);
                read(f, at);
                if (t + 1 < nt) multiply(f, e4m3, false, true);
                free = at;
                at = at + 1 < S ? at + 1 : 0;
            }
            multiply(f, e4m3, part, counts);
        }
    };
    if constexpr (MAY_E4M3) {
        uint32_t any = 0;
#pragma unroll
        for (int i = 0; i < 8; i++) any |= halves[2 * i + 1];
        if (__builtin_amdgcn_readfirstlane(any)) walk(std::false_type{});
        else walk(std::true_type{});
    } else walk(std::false_type{});
    wait_copies<0>();
    __syncthreads();   // the ring makes room for the sums

    // The waves' sums over k, 8 KB of each wave at a time.  A quad: n = LC (CB wn + j) + 8 e + 4 qh .. + 3, m = LC b + c (16 x 16: n = 4 qh ..);
    // lane l's lies at l ^ (its number), so that threads can take a row's quads one after the other.
    float* const red = (float*)smem;
    constexpr int PIECES = CB * E4;   // of a round, which is a row block
#pragma unroll
    for (int rd = 0; rd < RB; rd++) {
#pragma unroll
        for (int j = 0; j < CB; j++)
#pragma unroll
            for (int e = 0; e < E4; e++) {
                v4f v;
                if constexpr (BIG) v = (v4f){acc[j][rd][4 * e], acc[j][rd][4 * e + 1], acc[j][rd][4 * e + 2], acc[j][rd][4 * e + 3]};
                else v = acc[j][rd];
                const int piece = j * E4 + e;
                *(v4f*)(red + (wave * PIECES + piece) * 256 + 4 * (lane ^ (BIG ? 2 * piece + qh : 4 * piece + qh))) = v;
            }
        __syncthreads();
        constexpr int QUADS = WW_COLS / 4;   // of a row
#pragma unroll
        for (int i = 0; i < LC * QUADS / 512; i++) {
            const int t = tid + 512 * i, nq = t % QUADS, ml = t / QUADS;
            const int w_n = nq / (CB * LC / 4), in = nq % (CB * LC / 4);
            const int piece = BIG ? in >> 1 : in >> 2, half = BIG ? in & 1 : in & 3;
            const int slot = (half * LC + ml) ^ (BIG ? 2 * piece + half : 4 * piece + half);
            v4f sum = *(const v4f*)(red + (w_n * PIECES + piece) * 256 + 4 * slot);
#pragma unroll
            for (int h = 1; h < KW; h++) sum = sum + *(const v4f*)(red + ((h * WN + w_n) * PIECES + piece) * 256 + 4 * slot);
            const int m = m0 + LC * rd + ml, n = n0 + 4 * nq;
            if (m < Mi && n < Ni) {
                const int cols = Ni - n < 4 ? Ni - n : 4;
                if (splits > 1) {
                    float* dst = p.part + ((int64_t)blockIdx.y * Mi + m) * Ni + n;
                    if (cols == 4) __builtin_memcpy(dst, &sum, 16);
                    else {
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            if (e < cols) dst[e] = sum[e];
                    }
                } else {
                    uint16_t o[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        float v = sum[e];
                        if (p.bias) v = v + load_scalar_as_f32(p.bias, p.bias_dt, n + (e < cols ? e : cols - 1));
                        o[e] = bits_x<XDT>(v);
                    }
                    uint16_t* dst = p.y + (int64_t)m * Ni + n;
                    if (cols == 4) __builtin_memcpy(dst, o, 8);
                    else {
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            if (e < cols) dst[e] = o[e];
                    }
                }
            }
        }
        if (rd + 1 < RB) __syncthreads();
    }
}

struct WqWidePlan {
    int mb = 2, splits = 1, groups = 1;
    bool kn = false, dwords = false;   // [K, N] storage; its rows are no whole 16-byte pieces
    float us = 0.0f;
};

template <int XDT, int WBITS, int MB, bool HAS_OFF, int STORAGE>
int launch_one(const WqParams& p, const WqWidePlan& pl, hipStream_t st)
{
    auto k = wq_wide_kernel<XDT, WBITS, MB, HAS_OFF, STORAGE>;
    static std::atomic<uint64_t> attr_set{0};   // one bit per device: the attribute belongs to the (kernel, device) pair
    if (!device_flag_test(attr_set)) {
        hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, 163840);
        if (e != hipSuccess) return (int)e;
        device_flag_set(attr_set);
    }
    const int tiles = (int)((p.K + WW_KT - 1) / WW_KT);
    const dim3 grid((unsigned)((p.N + WW_COLS - 1) / WW_COLS), (unsigned)pl.splits, (unsigned)((p.M + 16 * MB - 1) / (16 * MB)));
    note_route("wq_wide", pl.splits);
    hipLaunchKernelGGL(k, grid, dim3(512), ww_ring(WBITS, MB) + pl.groups * WW_COLS * 4, st, p, tiles, pl.splits, pl.groups);
    if (hipError_t e = hipGetLastError(); e != hipSuccess || pl.splits == 1) return (int)e;
    launch_wq_splitk_reduce(p, pl.splits, XDT, st);
    return (int)hipGetLastError();
}
template <int XDT, int WBITS, bool HAS_OFF, int STORAGE>
int launch_mb(const WqParams& p, const WqWidePlan& pl, hipStream_t st)
{
    if (pl.mb == 1) return launch_one<XDT, WBITS, 1, HAS_OFF, STORAGE>(p, pl, st);
    if (pl.mb == 2) return launch_one<XDT, WBITS, 2, HAS_OFF, STORAGE>(p, pl, st);
    if (pl.mb == 4) return launch_one<XDT, WBITS, 4, HAS_OFF, STORAGE>(p, pl, st);
    return launch_one<XDT, WBITS, 8, HAS_OFF, STORAGE>(p, pl, st);
}
template <int XDT, int WBITS>
int launch_form(const WqParams& p, const WqWidePlan& pl, hipStream_t st)
{
    if (!pl.kn) return p.offset ? launch_mb<XDT, WBITS, true, WW_NK>(p, pl, st) : launch_mb<XDT, WBITS, false, WW_NK>(p, pl, st);
    if (!pl.dwords) return p.offset ? launch_mb<XDT, WBITS, true, WW_KN>(p, pl, st) : launch_mb<XDT, WBITS, false, WW_KN>(p, pl, st);
    return p.offset ? launch_mb<XDT, WBITS, true, WW_KN4>(p, pl, st) : launch_mb<XDT, WBITS, false, WW_KN4>(p, pl, st);
}

// Which layout is best: what a launch takes, in us, the weight from memory, fitted to 1460 timed launches of 160 calls (M 1 .. 400, K 1024 .. 18432, N 1024 .. 28672; median error 5 %):
// workgroups one a CU, in rounds, their K tiles by type and row blocks, the scale table, the weight's stream as the other bound, the
// outputs, and the second kernel of a K split.
float wide_us(const OpsnnWqmmArgs& a, int wbits, bool kn, int mb, int splits, int64_t groups)
{
    static const float per_tile[2][2][2] = {{{0.257f, 0.354f}, {0.403f, 0.69f}}, {{0.379f, 0.42f}, {0.412f, 0.6f}}};   // [8 bits][bf16][offset]
    const int64_t strips = (a.N + WW_COLS - 1) / WW_COLS, tiles = (a.K + WW_KT - 1) / WW_KT, slabs = (a.M + 16 * mb - 1) / (16 * mb);
    const float rounds = (float)((strips * slabs * splits + 255) / 256), seg = (float)((tiles + splits - 1) / splits);
    const float t = per_tile[wbits == 8][a.x_dtype == DT_BF16][a.offset != nullptr] + 0.075f * (float)mb + (kn ? 0.039f : 0.0f);
    const float cu = rounds * (seg * t + 2.1f + 0.27f * (float)mb + 0.057f * (float)groups), hbm = (float)a.N * (float)a.K * (float)wbits / (8e6f * 4.2f);
    const float most = cu > hbm ? cu : hbm, least = cu > hbm ? hbm : cu, q = least / most;
    const float out_m = (float)a.M * (float)a.N * 1e-6f;
    return 3.15f + 1.57f * out_m + most * (1.0f + 0.15f * q * q * q * q) + (splits > 1 ? 2.6f + 1.55f * (float)splits * out_m * (a.N % 4 ? 2.0f : 1.0f) : 0.0f);
}

bool wide_plan(const OpsnnWqmmArgs& a, const WqForm& f, WqWidePlan& pl)
{
    const int64_t strips = (a.N + WW_COLS - 1) / WW_COLS, tiles = (a.K + WW_KT - 1) / WW_KT;
    pl.us = 1e30f;
    auto consider = [&](int mb) {
        const int64_t slabs = (a.M + 16 * mb - 1) / (16 * mb);
        static const int steps[8] = {1, 2, 3, 4, 6, 8, 12, 16};
        for (int s : steps) {
            if (s > 1 && (tiles < 2 * s || strips * slabs * s > 1024)) break;
            const int64_t per = (tiles + s - 1) / s, g = f.group >= a.K ? 1 : (per * WW_KT + f.group - 1) / f.group + 1;
            if (g > ww_groups(f.wbits, mb)) continue;
            const float us = wide_us(a, f.wbits, pl.kn, mb, s, g);
            if (us < pl.us) { pl.us = us; pl.mb = mb; pl.splits = s; pl.groups = (int)g; }
        }
    };
    if (a.M <= 16) consider(1);
    else if (a.M <= 32) consider(2);
    else if (a.M <= 64) { consider(4); consider(2); }
    else { consider(8); consider(4); }
    return pl.us < 1e30f;
}

// Whether a call runs here at all: what the chosen layout typically takes (see wq_cost.h).  From 65 rows fitted to 937 calls of 65 .. 1024 (half of
// them for the fit, median error of the others 3 %); up to 64 rows to the kernel before its 32 x 32 x 16 products, whose times some calls are
// now a few percent below.
double wide_typical_us(const OpsnnWqmmArgs& a, int wbits, const WqWidePlan& pl)
{
    const int w8 = wbits == 8, bf = a.x_dtype == DT_BF16;
    const bool off = a.offset != nullptr;
    const int64_t strips = (a.N + WW_COLS - 1) / WW_COLS, tiles = (a.K + WW_KT - 1) / WW_KT, slabs = (a.M + 16 * pl.mb - 1) / (16 * pl.mb);
    const double out_m = (double)a.M * (double)a.N * 1e-6, mb = (double)pl.mb, mbytes = wq_typical_mb(wbits, a.N, a.K);
    const double rounds = (double)((strips * slabs * pl.splits + 255) / 256), steps = (double)((tiles + pl.splits - 1) / pl.splits);
    if (a.M > 64) {
        static const double tile[2][2] = {{0.175, 0.230}, {0.247, 0.282}}, offs[2] = {0.071, 0.241};   // [8 bits][bf16]
        const double t = tile[w8][bf] + (off ? offs[bf] : 0.0) + 0.0924 * mb + (pl.kn ? 0.0386 : 0.0) + (pl.dwords ? 0.0233 * wbits : 0.0);
        return 2.22 + 1.206 * out_m + wq_typical_both(rounds * (steps * t + 2.73 + 0.045 * mb + 0.0324 * pl.groups), mbytes / 6.86) +
               (pl.splits > 1 ? 3.82 + 1.247 * pl.splits * out_m : 0.0);
    }
    static const double tile[2][2][2] = {{{0.343, 0.444}, {0.486, 0.82}}, {{0.407, 0.502}, {0.449, 0.802}}};   // [8 bits][bf16][offset]
    const double t = tile[w8][bf][off] + 0.066 * mb + (pl.kn ? 0.056 : 0.0) + (pl.dwords ? 0.0125 * wbits : 0.0);
    return 2.39 + 1.33 * out_m + wq_typical_both(rounds * (steps * t + 1.91 + 0.355 * mb + 0.0143 * pl.groups), mbytes / 6.56) +
           (pl.splits > 1 ? 2.9 + 2.09 * pl.splits * out_m * (a.N % 4 ? 2.0 : 1.0) : 0.0);
}
// What the call typically takes on the kernel that it runs on otherwise.
double others_typical_us(const OpsnnWqmmArgs& a, const WqForm& f)
{
    if (a.M > 64) return wq_many_rows_typical_us(a);
    if (!f.nk) return wq_kn_wanted(a) ? wq_kn_typical_us(a) : 1e30;   // (else behind a re-layout)
    if (a.M <= 16 && f.stream && a.K % 128 == 0) {
        // up to 16 rows, whole chunks: x in registers, x whole in LDS, or the streaming kernel
        WqXregPlan x;
        const bool resx = a.K / (4 * (128 / f.wbits)) % 4 == 0 && (a.M + 1) * (a.K * 2 + 16) <= 65536;
        if (wq_xreg_plan(f.wbits, a.M, a.K, x) && (a.M >= 4 || (x.splits > 1 && !resx))) return x.splits == 1 ? 0.0 : wq_xreg_typical_us(a, f, x);
        return resx ? wq_resx_typical_us(a, f) : wq_stream_typical_us(a, f);
    }
    if (uint64_t bytes; wq_nk_wanted(a, &bytes)) return wq_nk_typical_us(a);
    if (f.rows && (a.M > 32 || wq_part_slices(f.wbits, a.M, a.N, a.K, f.group, true) > 1)) return wq_many_rows_typical_us(a);
    if (f.stream) return wq_stream_typical_us(a, f);
    return wq_general_counts(a, f) ? wq_general_typical_us(a) : 1e30;
}

// Does the call run here?  Looks at what both phases know: not at the weight's address (launch_wq_wide declines an unaligned one).
//
// Where the two estimates above say so, the weight from memory and in the last-level cache.  From 65 rows, of 1151 calls timed here, on the pass and
// on the other kernels 28 take 5 % longer than on the fastest, 6 by 10 %, the worst 1.19 times; with all estimates fitted to these kernels' former
// times 95 did, 52 by 10 %: 576 x 14336 x 14144 int8 280 us on the many-rows kernel, 328 here.  Up to 64 rows: profiles/weight_only_wide_rule.txt.
//
// Below 2^20 codes nothing was timed; from 65 rows the pass is ahead below 2^21 (189 x 1152 x 1088 12.1 there, 13.7 here).  Up to 16 rows:
// [K, N] storage not where the weight is large and wide, of 13 such calls seven 8 to 36 % faster there, one 12 % faster here (5 x 16256 x 25792 60 us there, 77
// here; 4 x 2560 x 27968 26.6 and 23.4), of 47 others none slower by the estimates than there, six that stay there 5 to 18 % faster here; [N, K] storage from 8 MB, and not where K is one whole shape of the x-in-registers kernel (16 x 8192 x 28672 36 there, 44 here;
// 4 x 3072 x 3128 7.3 and 10.5).  To 1024 rows (630 x 9472 x 18624 int4 fp16 326 -> 268,
// 707 x 9024 x 4160 int8 99 -> 77); of seven calls beyond one gained (1.07) and one lost (1534 x 1728 x 2184 21 -> 26).
//
// Rows in dwords: of 126 drawn calls of that kind 68 come here, 1.22 times as fast as on the pass and the [K, N] decode kernel: 156 x 7168 x 21520 int4 bf16 208 -> 100 us, 85 x 11008 x 2456 37 -> 21, 53 x 1408 x 22192 28 -> 15.
// Not where the estimates were wrong about them: from 257 rows with few k (510 x 1152 x 5744 21 there, 24 here), int8 up to 16 rows
// (10 x 13184 x 3944 20.7 and 22.0).
bool wide_wanted(const OpsnnWqmmArgs& a, WqWidePlan& pl)
{
    if ((a.w_dtype != DT_I4 && a.w_dtype != DT_I8) || (a.x_dtype != DT_F16 && a.x_dtype != DT_BF16)) return false;
    if (a.scale_dtype != a.x_dtype || a.force_variant != 0 || (uintptr_t)a.x % 16 != 0) return false;
    if (a.M > 1024 || a.K % 32 != 0 || a.K < 256 || a.N < 256 || a.K >= (1ll << 23) || a.N >= (1ll << 24)) return false;
    if (opsnn_wq_tile_min() <= 128 || !opsnn_wq_narrow_slabs()) return false;   // (test hooks of the other kernels)
    const WqForm f = wq_form(a);
    const int64_t codes = a.N * a.K;
    pl.kn = !f.nk;
    if (pl.kn && (a.w.col_stride != 1 || a.w.row_stride != a.N || a.N % (32 / f.wbits) != 0)) return false;
    pl.dwords = pl.kn && a.N % (128 / f.wbits) != 0;
    if (pl.dwords && ((a.M > 256 && a.K < 1536) || (a.M <= 16 && f.wbits == 8))) return false;
    if (f.group < a.K && (f.group < 32 || (f.group & (f.group - 1)) != 0)) return false;
    if (codes < (a.M > 64 ? 1ll << 21 : 1ll << 20)) return false;
    if (pl.kn && a.w_dtype == DT_I8 && a.M <= 16 && codes <= (1ll << 24)) return false;   // (as in wq_kn.hip)
    if (a.M <= 16 && (pl.kn ? codes > (1ll << 26) && a.N > 6144 : codes * f.wbits < (1ll << 26))) return false;
    return wide_plan(a, f, pl) && wide_typical_us(a, f.wbits, pl) < others_typical_us(a, f);
}
}  // namespace

static uint64_t wide_bytes(const OpsnnWqmmArgs& a, const WqWidePlan& pl)
{
    return pl.splits > 1 ? ((uint64_t)pl.splits * (uint64_t)a.M * (uint64_t)a.N * 4 + 255) / 256 * 256 : 0;
}
static bool is_kn(const OpsnnWqmmArgs& a) { return a.w.row_stride != 1 && a.w.col_stride == 1 && a.w.row_stride == a.N; }
static OpsnnWqmmArgs as_nk(OpsnnWqmmArgs a)
{
    a.w.row_stride = 1; a.w.col_stride = a.K;
    return a;
}
// ([K, N] storage: also what the call needs on a K-contiguous copy from the weight cache, which only phase 2 knows of)
bool wq_wide_wanted(const OpsnnWqmmArgs& a, uint64_t* workspace)
{
    WqWidePlan pl;
    const bool here = wide_wanted(a, pl);
    *workspace = here ? wide_bytes(a, pl) : 0;
    if (is_kn(a)) {
        const OpsnnWqmmArgs b = as_nk(a);
        if (WqWidePlan plb; wide_wanted(b, plb)) {
            const uint64_t bytes = wide_bytes(b, plb);
            if (bytes > *workspace) *workspace = bytes;
            return true;
        }
    }
    return here;
}
int launch_wq_wide(const OpsnnWqmmArgs& a0, hipStream_t st)
{
    OpsnnWqmmArgs a = a0;
    WqWidePlan pl;
    if (is_kn(a) && weight_cache_on()) {   // a caller who keeps K-contiguous copies gets the bits of that form, from here or from the kernels behind
        const OpsnnWqmmArgs b = as_nk(a);
        if (!wide_wanted(b, pl) || (pl.splits > 1 && !a.workspace)) return OPSNN_NOT_TAKEN;
        if (const void* copy = weight_cache_get(a.w.ptr, a.K, a.N, a.w_dtype == DT_I4 ? 4 : 8, 1, st)) { a = b; a.w.ptr = copy; }
    }
    if ((uintptr_t)a.w.ptr % 16 != 0 || !wide_wanted(a, pl) || (pl.splits > 1 && !a.workspace)) return OPSNN_NOT_TAKEN;
    const int wbits = a.w_dtype == DT_I4 ? 4 : 8;
    WqParams p{};
    p.group = a.group > 0 && a.group < a.K ? a.group : a.K;
    p.x = (const uint16_t*)a.x;
    p.w = (const uint8_t*)a.w.ptr; p.ldw = (pl.kn ? a.w.row_stride : a.w.col_stride) * wbits / 8;
    p.scale = (const uint16_t*)a.scale.ptr; p.offset = (const uint16_t*)a.offset;
    p.s_rs = a.scale.row_stride; p.s_cs = a.scale_n == 1 ? 0 : a.scale.col_stride;
    p.bias = a.bias; p.bias_dt = a.bias_dtype;
    p.y = (uint16_t*)a.y; p.M = a.M; p.N = a.N; p.K = a.K;
    p.group_shift = p.group >= p.K ? 31 : __builtin_ctzll((unsigned long long)p.group);
    p.part = (float*)a.workspace;
    if (a.x_dtype == DT_F16) return wbits == 4 ? launch_form<DT_F16, 4>(p, pl, st) : launch_form<DT_F16, 8>(p, pl, st);
    return wbits == 4 ? launch_form<DT_BF16, 4>(p, pl, st) : launch_form<DT_BF16, 8>(p, pl, st);
}

}  // namespace opsnn
