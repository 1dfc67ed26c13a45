// Weight-only matmul, up to 512 rows of x, either storage of the weight ([N, K] and [K, N]), any group that is a power of two from 32.
//
// What bounded these calls (17 .. 64 rows on the kernels of wq_nk.hip, wq_kn.hip and wqmm_stream.hip.h, more rows on the dequantising
// pass of wq_dense.hip): operands loaded straight into the layout of the matrix instructions, 16 rows per 16 lanes, take 66 clocks a KB
// in the memory pipeline of a CU, twice what the same bytes take with neighbouring lanes side by side; and a dequantised copy of the
// weight is four times its bytes, written and read.  So weight and x travel global -> LDS as they lie, 16 bytes a lane, asynchronously,
// in K tiles of 128 for 128 columns and 16 MB rows, through a ring of as many stages as the LDS holds, one barrier a tile, and every
// weight is dequantised once per 16 MB rows, in registers.
//
// Eight waves: two halves of the columns times four steps of 32 k.  A wave multiplies 64 columns (four blocks of 16) by all rows, so
// that a fragment of x serves four column blocks; the four sums over k meet in LDS at the end, in order.  blockIdx.y cuts K further
// (fp32 partial sums, added in order by wq_splitk_reduce_kernel), blockIdx.z takes further slabs of 16 MB rows.  The scales of the
// workgroup's columns lie in LDS as a table, laid down once: a compiler's load in the loop would be waited for with every copy under
// way.
//
// What bounds it now is the issue of vector instructions: dequantising takes some 20 per 8 weights of a lane, two of which a matrix
// instruction hides (mfma_16x16x32 7.2 ns with none or two of them behind it, 18 with eight).  [K, N] storage: two rows of k of one
// column share a dword once their 16-bit pieces are joined, so the splice delivers pairs in k order and x needs no permutation;
// [N, K] storage permutes x.
//
// LDS rows, conflict-free for the reads below: x 256 bytes, 16-byte chunk c of row r at c ^ (r % 16); [N, K] weights 64 bytes (4 bits),
// c ^ (r / 4 % 4), or 128, c ^ (r / 2 % 8); [K, N] weights 64 bytes, row k at slot k ^ (k / 8 % 4), or 128, slot k ^ (k / 8 % 2) with
// the halves swapped where k / 16 is odd.
//
// Measured, the weight from memory, a call before and now: [K, N] int4, 110 x 11008 x 24768 fp16 346 -> 126 us, 73 x 6656 x 2752 34.9 -> 19.0,
// 200-row slabs 195 x 7296 x 15680 154 -> 83, int8 67 x 3840 x 12864 65 -> 30; [N, K] int4 57 x 9856 x 24349 98 -> 63, 37 x 7936 x 8576 bf16 69 -> 33,
// int8 118 x 14336 x 8512 bf16 135 -> 58; 341 drawn calls of 1 .. 600 rows 1.21 times as fast.
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

// [K, N] storage: two rows of k of column j -> a pair of values of x's type.  4 bits: w0 holds four columns of both rows; 8 bits: of one
// row each.  The arithmetic and its roundings are dequant8's.
template <int XDT, int WBITS, bool HAS_OFF>
__device__ __forceinline__ int kn_pair(uint32_t w0, uint32_t w1, int j, uint32_t so, const DqConst& dc)
{
    if constexpr (XDT == DT_F16) {
        const _Float16 sh = __builtin_bit_cast(_Float16, (uint16_t)so), oh = __builtin_bit_cast(_Float16, (uint16_t)(so >> 16));
        h2 t;
        if constexpr (WBITS == 4) {
            const uint32_t q = j >= 2 ? w0 >> 8 : w0;
            const h2 c1032 = {(_Float16)-1032.0f, (_Float16)-1032.0f}, c72 = {(_Float16)-72.0f, (_Float16)-72.0f}, r16 = {(_Float16)0.0625f, (_Float16)0.0625f};
            if (j & 1) t = __builtin_elementwise_fma(__builtin_bit_cast(h2, (q & dc.mhi) ^ dc.chi), r16, c72);
            else t = __builtin_bit_cast(h2, (q & dc.mlo) ^ dc.clo) + c1032;
        } else {
            const h2 c1152 = {(_Float16)-1152.0f, (_Float16)-1152.0f};
            t = __builtin_bit_cast(h2, __builtin_amdgcn_perm(w1, w0, 0x0c000c00u | (uint32_t)j | (uint32_t)(4 + j) << 16) ^ 0x64806480u) + c1152;
        }
        if constexpr (HAS_OFF) t = t + (h2){oh, oh};
        return (int)u32(t * (h2){sh, sh});
    } else {
        const float sc = bf16_to_f32((uint16_t)so), off = bf16_to_f32((uint16_t)(so >> 16));
        float a, b;
        if constexpr (WBITS == 4) {   // (16 times the weight, see dequant8)
            const uint32_t n = j & 1 ? w0 & 0xf0f0f0f0u : (w0 << 4) & 0xf0f0f0f0u;
            a = (float)((int)(n << (24 - 8 * (j >> 1))) >> 24);
            b = (float)((int)(n << (8 - 8 * (j >> 1))) >> 24);
        } else {
            a = (float)((int)(w0 << (24 - 8 * j)) >> 24);
            b = (float)((int)(w1 << (24 - 8 * j)) >> 24);
        }
        float s = sc;
        if constexpr (HAS_OFF) {
            const float one = WBITS == 4 ? 0.0625f : 1.0f;
            const uint32_t pk = pack2_bf16((v2f){__builtin_fmaf(a, one, off), __builtin_fmaf(b, one, off)});
            a = u2f(pk << 16);
            b = u2f(pk & 0xffff0000u);
        } else if constexpr (WBITS == 4) s = 0.0625f * sc;
        return (int)pack2_bf16((v2f){a * s, b * s});
    }
}

// bytes of a tile, stages of the ring, bytes of the ring (at least what the sums need at the end), groups that the table has room for
constexpr int ww_tile(int wbits, int mb) { return mb * 4096 + WW_COLS * WW_KT * wbits / 8; }
constexpr int ww_stages(int wbits, int mb)
{
    return wbits == 4 ? (mb <= 2 ? 6 : mb <= 4 ? 4 : 3) : (mb <= 4 ? 4 : 3);
}
constexpr int ww_ring(int wbits, int mb) { const int a = ww_tile(wbits, mb) * ww_stages(wbits, mb); return a > 65536 ? a : 65536; }
constexpr int ww_groups(int wbits, int mb) { return (163840 - ww_ring(wbits, mb)) / (WW_COLS * 4); }

template <int XDT, int WBITS, int MB, bool HAS_OFF, bool KN>
__global__ __launch_bounds__(512, 1) void wq_wide_kernel(WqParams p, int tiles, int splits, int gmax)
{
    constexpr int NB = 4, TILE = ww_tile(WBITS, MB), S = ww_stages(WBITS, MB);
    constexpr int XC = MB > 2 ? MB / 2 : 1, WC = WBITS / 4, CPT = XC + WC;   // copies per wave and tile
    constexpr int WROW = WW_KT * WBITS / 8;                                  // bytes of a weight row in a tile
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave & 1, kw = wave >> 1;
    const int r = lane & 15, q = lane >> 4;
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
        const int row = WBITS == 4 ? wave * 16 + (lane >> 2) : (wave * 2 + i) * 8 + (lane >> 3);
        if constexpr (KN) {
            // a tile row is a row of k; row k lies at slot k ^ (k / 8 % 4) (8 bits: k ^ (k / 8 % 2), and its halves swapped where k / 16 is odd)
            const int k = WBITS == 4 ? row ^ ((row >> 3) & 3) : row ^ ((row >> 3) & 1);
            const int c = WBITS == 4 ? (lane & 3) : (lane & 7) ^ (((row >> 4) & 1) << 2);
            const int at = 16 * c, last = (Ni - n0) * WBITS / 8 - 16;
            wo[i] = (uint32_t)k * (uint32_t)p.ldw + (at < last ? at : last);
        } else {
            const int n = n0 + row < Ni ? row : Ni - 1 - n0;
            const int c = WBITS == 4 ? (lane & 3) ^ ((row >> 2) & 3) : (lane & 7) ^ ((row >> 1) & 7);
            wo[i] = (uint32_t)n * (uint32_t)p.ldw + 16 * c;
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
        for (int i = 0; i < WC; i++) copy16_sbase(wbase + (KN ? k * p.ldw : k * WBITS / 8), wo[i], at + MB * 4096 + (wave * WC + i) * 1024);
#pragma unroll
        for (int i = 0; i < XC; i++) copy16_sbase(xbase + k * 2, xo[i], at + ((wave * XC + i) * 1024) % (MB * 4096));
    };

    v4f acc[NB][MB];
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
        for (int b = 0; b < MB; b++) acc[j][b] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
    const DqConst dqc = make_dq_const();
    uint32_t* const tab = (uint32_t*)(smem + ww_ring(WBITS, MB));
    struct Frags {
        v4i x[MB];
        uint32_t w[KN ? 8 : WBITS == 4 ? NB : 2 * NB];   // NK: column j's 8 codes; KN: row i of four columns
        uint32_t so[NB];
    };
    auto read = [&](Frags& f, int stage) {
        const int k = k_read < k_last ? k_read : k_last;
        k_read += WW_KT;
        const char* const at = smem + stage * TILE;
#pragma unroll
        for (int b = 0; b < MB; b++) f.x[b] = *(const v4i*)(at + (16 * b + r) * 256 + 16 * ((4 * kw + q) ^ r));
        if constexpr (KN && WBITS == 4) {
#pragma unroll
            for (int i = 0; i < 4; i++) {   // (row 32 kw + 8 q + i at the slot with i ^ q)
                const char* const a = at + MB * 4096 + (32 * kw + 8 * q) * 64 + 32 * wn + 2 * r;
                f.w[2 * i] = *(const uint16_t*)(a + ((2 * i) ^ q) * 64);
                f.w[2 * i + 1] = *(const uint16_t*)(a + ((2 * i + 1) ^ q) * 64);
            }
        } else if constexpr (KN) {
#pragma unroll
            for (int i = 0; i < 8; i++) f.w[i] = *(const uint32_t*)(at + MB * 4096 + (32 * kw + 8 * q + (i ^ (q & 1))) * 128 + 64 * (wn ^ (q >> 1)) + 4 * r);
        } else {
#pragma unroll
            for (int j = 0; j < NB; j++) {
                const char* const row = at + MB * 4096 + (wn * 64 + 16 * j + r) * WROW;
                if constexpr (WBITS == 4) f.w[j] = *(const uint32_t*)(row + 16 * (kw ^ (r >> 2)) + 4 * q);
                else __builtin_memcpy(f.w + 2 * j, __builtin_assume_aligned(row + 16 * ((2 * kw + (q >> 1)) ^ (r >> 1)) + 8 * (q & 1), 8), 8);
            }
        }
        const int g = group_at(k + 32 * kw) - g_lo;
#pragma unroll
        for (int j = 0; j < NB; j++) f.so[j] = tab[g * WW_COLS + wn * 64 + (KN ? 4 * r + j : 16 * j + r)];
    };
    auto multiply = [&](const Frags& f) {
        v4i xh[MB];
        uint32_t pairs[4];   // KN, 4 bits: rows 2 i, 2 i + 1 of four columns
        if constexpr (KN && WBITS == 4) {
#pragma unroll
            for (int i = 0; i < 4; i++) pairs[i] = f.w[2 * i] | f.w[2 * i + 1] << 16;
        }
#pragma unroll
        for (int b = 0; b < MB; b++) {
            xh[b] = f.x[b];
            if constexpr (WBITS == 4 && !KN) {   // halves [0..7] -> [0,4,1,5,2,6,3,7]
                const uint32_t a0 = (uint32_t)xh[b][0], a1 = (uint32_t)xh[b][1], a2 = (uint32_t)xh[b][2], a3 = (uint32_t)xh[b][3];
                xh[b] = (v4i){(int)__builtin_amdgcn_perm(a2, a0, 0x05040100u), (int)__builtin_amdgcn_perm(a2, a0, 0x07060302u),
                              (int)__builtin_amdgcn_perm(a3, a1, 0x05040100u), (int)__builtin_amdgcn_perm(a3, a1, 0x07060302u)};
            }
        }
#pragma unroll
        for (int j = 0; j < NB; j++) {
            v4i a;
            if constexpr (KN) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    if constexpr (WBITS == 4) a[i] = kn_pair<XDT, 4, HAS_OFF>(pairs[i], 0, j, f.so[j], dqc);
                    else a[i] = kn_pair<XDT, 8, HAS_OFF>(f.w[2 * i], f.w[2 * i + 1], j, f.so[j], dqc);
                }
            } else {
                const v4i piece = {(int)f.w[WBITS == 4 ? j : 2 * j], WBITS == 8 ? (int)f.w[(2 * j + 1) % (2 * NB)] : 0, 0, 0};
                a = dequant8<XDT, WBITS, HAS_OFF>(piece, 0, (uint16_t)f.so[j], (uint16_t)(f.so[j] >> 16), dqc);
            }
#pragma unroll
            for (int b = 0; b < MB; b++) {
                if constexpr (XDT == DT_F16) acc[j][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, xh[b]), acc[j][b], 0, 0, 0);
                else acc[j][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, xh[b]), acc[j][b], 0, 0, 0);
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
    auto store8 = [&](const Eight& v, int i) {
        const int g = t_g + 32 * i - g_lo;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const int ge = g + (by_group ? e : 0), ne = t_col + (by_group ? 0 : e);
            if (ge >= 0 && ge < gmax) tab[ge * WW_COLS + ne] = HAS_OFF ? v.s[e] | (uint32_t)v.o[e] << 16 : v.s[e];
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
    wait_copies<(S - 1) * CPT>();
    __syncthreads();
    const bool rest = base_of(nt - 1) + 32 * kw >= (t0 + nt - 1) * WW_KT;   // (a partial tile: the others were counted with the one before)
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
            multiply(now);
        };
        for (; t + 2 < nt; t += 2) {
            step(f0, f1);
            step(f1, f0);
        }
        if (t + 1 < nt) {
            step(f0, f1);
            if (rest) multiply(f1);
        } else if (rest) multiply(f0);
    } else {   // (no registers for a second set of fragments: tile t + S - 1 goes where tile t - 1 was)
        Frags f;
        int at = 0, free = S - 1;
        for (int t = 0; t < nt; t++) {
            wait_copies<(S - 2) * CPT>();
            __builtin_amdgcn_s_barrier();
            asm volatile("" : : : "memory");
            if (t > 0) issue(free);
            read(f, at);
            if (t + 1 < nt || rest) multiply(f);
            free = at;
            at = at + 1 < S ? at + 1 : 0;
        }
    }
    wait_copies<0>();
    __syncthreads();   // the ring makes room for the sums

    // acc[j][b][e]: n = n0 + 64 wn + 16 j + 4 q + e (KN: 4 (4 q + e) + j), m = m0 + 16 b + r, over the k of kw
    float* const red = (float*)smem;
#pragma unroll
    for (int b0 = 0; b0 < MB; b0 += 2) {
        constexpr int RB = MB < 2 ? 1 : 2;
#pragma unroll
        for (int j = 0; j < NB; j++)
#pragma unroll
            for (int b = 0; b < RB; b++) *(v4f*)(red + ((kw * 2 + wn) * (NB * RB) + j * RB + b) * 256 + lane * 4) =
                KN ? (v4f){acc[0][b0 + b][j], acc[1][b0 + b][j], acc[2][b0 + b][j], acc[3][b0 + b][j]} : acc[j][b0 + b];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < RB; i++) {
            const int t = tid + 512 * i, blk = t >> 6;   // block (wn, j, b)
            v4f sum = *(const v4f*)(red + t * 4);
#pragma unroll
            for (int h = 1; h < 4; h++) sum = sum + *(const v4f*)(red + (h * 2 * NB * RB) * 256 + t * 4);
            const int m = m0 + 16 * (b0 + blk % RB) + (t & 15), n = n0 + 64 * (blk / (NB * RB)) + (KN ? 4 : 16) * (blk / RB % NB) + (KN ? 16 : 4) * ((t >> 4) & 3);
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
        if (b0 + 2 < MB) __syncthreads();
    }
}

struct WqWidePlan {
    int mb = 2, splits = 1, groups = 1;
    bool kn = false;
    float us = 0.0f;
};

template <int XDT, int WBITS, int MB, bool HAS_OFF, bool KN>
int launch_one(const WqParams& p, const WqWidePlan& pl, hipStream_t st)
{
    auto k = wq_wide_kernel<XDT, WBITS, MB, HAS_OFF, KN>;
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
template <int XDT, int WBITS, bool HAS_OFF>
int launch_mb(const WqParams& p, const WqWidePlan& pl, hipStream_t st)
{
    if (pl.kn) {
        if (pl.mb == 1) return launch_one<XDT, WBITS, 1, HAS_OFF, true>(p, pl, st);
        if (pl.mb == 2) return launch_one<XDT, WBITS, 2, HAS_OFF, true>(p, pl, st);
        if (pl.mb == 4) return launch_one<XDT, WBITS, 4, HAS_OFF, true>(p, pl, st);
        return launch_one<XDT, WBITS, 8, HAS_OFF, true>(p, pl, st);
    }
    if (pl.mb == 1) return launch_one<XDT, WBITS, 1, HAS_OFF, false>(p, pl, st);
    if (pl.mb == 2) return launch_one<XDT, WBITS, 2, HAS_OFF, false>(p, pl, st);
    if (pl.mb == 4) return launch_one<XDT, WBITS, 4, HAS_OFF, false>(p, pl, st);
    return launch_one<XDT, WBITS, 8, HAS_OFF, false>(p, pl, st);
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

// Whether a call runs here at all: what the chosen layout typically takes (median error 3 %; see wq_cost.h).
double wide_typical_us(const OpsnnWqmmArgs& a, int wbits, const WqWidePlan& pl)
{
    static const double tile[2][2][2] = {{{0.343, 0.444}, {0.486, 0.82}}, {{0.407, 0.502}, {0.449, 0.802}}};   // [8 bits][bf16][offset]
    const int64_t strips = (a.N + WW_COLS - 1) / WW_COLS, tiles = (a.K + WW_KT - 1) / WW_KT, slabs = (a.M + 16 * pl.mb - 1) / (16 * pl.mb);
    const double t = tile[wbits == 8][a.x_dtype == DT_BF16][a.offset != nullptr] + 0.066 * pl.mb + (pl.kn ? 0.056 : 0.0), out_m = (double)a.M * (double)a.N * 1e-6;
    const double cu = (double)((strips * slabs * pl.splits + 255) / 256) * ((double)((tiles + pl.splits - 1) / pl.splits) * t + 1.91 + 0.355 * pl.mb + 0.0143 * pl.groups);
    return 2.39 + 1.33 * out_m + wq_typical_both(cu, wq_typical_mb(wbits, a.N, a.K) / 6.56) + (pl.splits > 1 ? 2.9 + 2.09 * pl.splits * out_m * (a.N % 4 ? 2.0 : 1.0) : 0.0);
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
// Where the two estimates above say so.  (Of 2989 calls, 1797 of them drawn after the fit, timed on either side with the weight from memory and in
// the last-level cache, 1983 run here, 46 of them 5 % slower or more than there, 14 by 10 %, the worst 1.28 times; among other fitted ones the
// worst is 1.4, 339 x 15872 x 12160 bf16 x int8 226 us, 162 on the many-rows kernel.  Before there were estimates for [K, N] storage and up to 16
// rows, and with the other estimates fitted to the weight from memory, 153 were, 82 by 10 %: 491 x 8448 x 2112 [K, N] int8 48 us with the pass
// and 75 here, 27 x 17920 x 25376 [K, N] bf16 124 and 156, 3 x 1536 x 13184 bf16 10.7 and 13.6, 18 x 3328 x 1152 bf16 x int8 9.8 and 11.1.)
//
// Below 2^20 codes nothing was timed; from 65 rows the pass is ahead below 2^21 (189 x 1152 x 1088 12.1 there, 13.7 here).  Up to 16 rows:
// [K, N] storage not where the weight is large and wide, of 68 such calls 56 faster there (16 x 8192 x 28672 40.7 us, 47.9 here; 5 x 12288 x 27072 61
// and 86); [N, K] storage from 8 MB, and not where K is one whole shape of the x-in-registers kernel (16 x 8192 x 28672 36 there, 44 here;
// 4 x 3072 x 3128 7.3 and 10.5).  From 513 rows the dequantising pass is ahead of a fifth slab.
bool wide_wanted(const OpsnnWqmmArgs& a, WqWidePlan& pl)
{
    if ((a.w_dtype != DT_I4 && a.w_dtype != DT_I8) || (a.x_dtype != DT_F16 && a.x_dtype != DT_BF16)) return false;
    if (a.scale_dtype != a.x_dtype || a.force_variant != 0 || (uintptr_t)a.x % 16 != 0) return false;
    if (a.M > 512 || a.K % 32 != 0 || a.K < 256 || a.N < 256 || a.K >= (1ll << 23) || a.N >= (1ll << 24)) return false;
    if (opsnn_wq_tile_min() <= 128 || !opsnn_wq_narrow_slabs()) return false;   // (test hooks of the other kernels)
    const WqForm f = wq_form(a);
    const int64_t codes = a.N * a.K;
    pl.kn = !f.nk;
    if (pl.kn && (a.w.col_stride != 1 || a.w.row_stride != a.N || a.N % (128 / f.wbits) != 0)) return false;
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
    if (a.x_dtype == DT_F16) {
        if (wbits == 4) return a.offset ? launch_mb<DT_F16, 4, true>(p, pl, st) : launch_mb<DT_F16, 4, false>(p, pl, st);
        return a.offset ? launch_mb<DT_F16, 8, true>(p, pl, st) : launch_mb<DT_F16, 8, false>(p, pl, st);
    }
    if (wbits == 4) return a.offset ? launch_mb<DT_BF16, 4, true>(p, pl, st) : launch_mb<DT_BF16, 4, false>(p, pl, st);
    return a.offset ? launch_mb<DT_BF16, 8, true>(p, pl, st) : launch_mb<DT_BF16, 8, false>(p, pl, st);
}

}  // namespace opsnn
